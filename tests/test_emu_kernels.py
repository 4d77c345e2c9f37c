"""CPU checks of the HIP kernel sources themselves, compiled for the host against a fiber-based stand-in
for the HIP runtime (tests/emu).  Same operators, same C ABI, same oracle as the GPU parity tests, on
small shapes; buffers sit against guard pages so an out-of-range index is a SIGSEGV here rather than a
GPU fault.  The shipped library is not involved: these tests prove indexing/synchronisation logic, the
`-m gpu` tests prove the device build."""
import pytest
import torch

from mindspeed_mm_amd._lib import kernel_timings, ptr
from tests import parity as P
from tests.emu.emu_backend import emu_ops, guarded, guarded_outputs

BF, F32 = torch.bfloat16, torch.float32


@pytest.fixture(scope="module")
def ops():
    return emu_ops()


@pytest.fixture(autouse=True)
def _outputs_against_guard_pages():
    """Every test here also runs with what the operators allocate themselves (outputs, gradients, workspaces)
    flush against guard pages, not only the inputs the test hands in."""
    with guarded_outputs():
        yield


@pytest.mark.parametrize("dtype,B,T,Hqk,Hv,K,V", [
    (F32, 2, 3, 1, 2, 64, 64), (BF, 2, 2, 2, 4, 128, 128), (F32, 1, 1, 1, 1, 128, 192), (BF, 1, 4, 1, 2, 256, 128),
])
def test_recurrent(ops, dtype, B, T, Hqk, Hv, K, V):
    P.check_recurrent(ops, "cpu", B, T, Hqk, Hv, K, V, dtype, wrap=guarded)
    P.check_recurrent(ops, "cpu", B, T, Hqk, Hv, K, V, dtype, l2=False, with_state=False, wrap=guarded)


@pytest.mark.parametrize("dtype,K", [(BF, 64), (BF, 128), (BF, 256), (F32, 128)])
def test_recurrent_rows_on_any_element(ops, dtype, K):
    """q and k may start on any element: the kernel's loads are wider than one, but promise no more alignment than that."""
    x = P.gdn_inputs(2, 2, 1, 2, K, 64, dtype, seed=2)
    want = ops.fused_recurrent_gated_delta_rule(*(x[n] for n in ("q", "k", "v", "g", "beta")), initial_state=x["h0"],
                                                output_final_state=True, use_qk_l2norm_in_kernel=True)
    for n in ("q", "k"):
        x[n] = torch.cat([x[n].flatten()[:1], x[n].flatten()])[1:].view(x[n].shape)
        assert x[n].data_ptr() % 4 or dtype == F32 and x[n].data_ptr() % 8
    got = ops.fused_recurrent_gated_delta_rule(*(x[n] for n in ("q", "k", "v", "g", "beta")), initial_state=x["h0"],
                                               output_final_state=True, use_qk_l2norm_in_kernel=True)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype,K,V", [(BF, 128, 128), (BF, 128, 192), (F32, 64, 128), (BF, 256, 128)])
def test_recurrent_bits_do_not_depend_on_the_batch(ops, dtype, K, V):
    P.check_recurrent_batch_bits(ops, "cpu", (1, 9), 1, 1, K, V, dtype)   # fewer and more states than compute units


@pytest.mark.parametrize("dtype,T,cu,Hqk,Hv,K,V", [
    (F32, 12, [0, 3, 3, 8, 12], 1, 2, 64, 64), (BF, 9, [0, 1, 6], 1, 2, 128, 64),
])
def test_recurrent_packed_sequences(ops, dtype, T, cu, Hqk, Hv, K, V):
    P.check_recurrent_packed(ops, "cpu", T, cu, Hqk, Hv, K, V, dtype, wrap=guarded)
    P.check_recurrent_packed(ops, "cpu", T, cu, Hqk, Hv, K, V, dtype, l2=False, with_state=False, wrap=guarded)


@pytest.mark.parametrize("dtype,B,T,Hqk,Hv,K,V,l2,cu", [
    (F32, 1, 64, 1, 1, 64, 64, False, None),
    (F32, 2, 100, 2, 4, 128, 128, True, None),
    (BF, 1, 200, 1, 2, 128, 128, True, None),
    (BF, 1, 140, 2, 2, 64, 64, False, [0, 5, 70, 71, 140]),
    (BF, 1, 128, 1, 1, 128, 256, True, None),
    (F32, 1, 96, 1, 1, 128, 192, True, [0, 1, 38, 96]),
])
def test_chunk_forward(ops, dtype, B, T, Hqk, Hv, K, V, l2, cu):
    P.check_chunk(ops, "cpu", B, T, Hqk, Hv, K, V, dtype, l2=l2, cu=cu, wrap=guarded, h0_std=0.1)


@pytest.mark.parametrize("dtype,B,T,Hqk,Hv,K,V,l2,cu", [
    (F32, 1, 130, 1, 2, 64, 64, True, None),
    (F32, 2, 100, 2, 4, 128, 128, True, None),
    (BF, 1, 200, 1, 2, 128, 128, True, None),
    (BF, 1, 140, 2, 2, 64, 64, False, [0, 5, 70, 71, 140]),
    (F32, 1, 96, 1, 1, 128, 192, True, [0, 1, 38, 96]),
    (BF, 1, 100, 1, 6, 64, 64, True, None),          # more value heads per group than the prep kernel has waves
    (F32, 1, 70, 1, 3, 64, 64, True, [0, 3, 70]),
])
def test_chunk_backward(ops, dtype, B, T, Hqk, Hv, K, V, l2, cu):
    P.check_chunk(ops, "cpu", B, T, Hqk, Hv, K, V, dtype, l2=l2, cu=cu, backward=True, wrap=guarded, h0_std=0.1)


@pytest.mark.parametrize("cu", [[0, 0, 70], [0, 70, 70], [0, 30, 30, 100], [0, 0, 0, 64]])
def test_chunk_packed_with_empty_sequences(ops, cu):
    """A sequence of length 0 has no chunk: its final state is its initial state, its gradients are empty."""
    P.check_chunk(ops, "cpu", 1, cu[-1], 1, 2, 64, 64, F32, cu=cu, backward=True, wrap=guarded, h0_std=0.1)


@pytest.mark.parametrize("B,T,cu", [(0, 64, None), (1, 64, [0])])
def test_no_sequence_is_refused(ops, B, T, cu):
    """A batch without a sequence raises, in the sizes whose recurrences may be cut into segments too."""
    x = P.kda_inputs(1, T, 2, 128, 128, BF, N=1)
    r = {n: x[n][:B] for n in ("q", "k", "v", "g", "beta")}
    cu_t = torch.tensor(cu, dtype=torch.int64) if cu else None
    with pytest.raises(ValueError):
        ops.chunk_gated_delta_rule(r["q"], r["k"], r["v"], r["g"][..., 0].float(), r["beta"], cu_seqlens=cu_t)
    with pytest.raises(ValueError):
        ops.chunk_kda(r["q"], r["k"], r["v"], r["g"].float(), r["beta"], cu_seqlens=cu_t, A_log=x["A_log"],
                      dt_bias=x["dt_bias"], use_gate_in_kernel=True)


@pytest.mark.parametrize("dtype,B,T,Hqk,Hv,K,V,cu", [
    (BF, 1, 200, 1, 2, 128, 128, None), (F32, 1, 140, 1, 2, 64, 64, [0, 5, 70, 140]),
    (BF, 1, 135, 1, 2, 64, 192, [0, 5, 70, 135]),   # reverse recurrence with two loading waves, and with four
])
def test_chunk_backward_recompute_mode_equals_stored_mode(ops, dtype, B, T, Hqk, Hv, K, V, cu):
    P.check_chunk_recompute_equals_stored(ops, "cpu", B, T, Hqk, Hv, K, V, dtype, cu=cu, wrap=guarded, h0_std=0.1)


@pytest.mark.parametrize("T,Hqk,Hv,K,V,l2", [
    (70, 1, 3, 64, 128, True),     # three heads to a group, half of the waves without columns of K of their own
    (65, 1, 2, 128, 192, True),    # R in two parts, the second of two V blocks; a last chunk of one token
    (64, 1, 1, 128, 64, False),    # one pair of V blocks; no l2 norm
    (33, 1, 2, 64, 64, True),      # several heads and V = 64: the four-wave kernel
    (130, 2, 2, 64, 256, False),
])
def test_chunk_local_backward_of_head_groups(ops, T, Hqk, Hv, K, V, l2):
    """The chunk-local kernel where its tiles, its V blocks and the sums over a group's heads end."""
    P.check_chunk(ops, "cpu", 1, T, Hqk, Hv, K, V, BF, l2=l2, backward=True, wrap=guarded, h0_std=0.1, seed=5)


@pytest.mark.parametrize("dtype,V,launched", [
    (BF, 128, {"chunk_bwd_local16_kernel": 1}), (BF, 64, {"chunk_bwd_local_kernel": 2}), (F32, 128, {"chunk_bwd_local_kernel": 2}),
])
def test_chunk_local_backward_is_timed_under_its_kernels_name(ops, dtype, V, launched):
    """Two heads to a group: one launch of the eight-wave kernel, or one launch per head of the four-wave one."""
    ops.lib.gdn_profile_enable(1)
    try:
        P.check_chunk(ops, "cpu", 1, 64, 1, 2, 64, V, dtype, backward=True)
        assert {n: c for n, (_, c) in kernel_timings(ops.lib).items() if n.startswith("chunk_bwd_local")} == launched
    finally:
        ops.lib.gdn_profile_enable(0)


@pytest.mark.parametrize("K,V", [(128, 128), (64, 256)])
def test_group_sums_read_nothing_that_was_not_written(ops, monkeypatch, K, V):
    """The dq, dk sums that pass from head to head of a group hold the rows past a short last chunk's end too: with a
    workspace of NaN patterns these stay finite, as nothing they are formed of is left over from before."""
    import mindspeed_mm_amd.ops as M
    T, Hqk, Hv = 70, 1, 3
    parts, real = [], M._chunk_workspace

    def filled(*args):
        ws, nbytes = real(*args)
        parts.append(ws.fill_(0xff))
        return ws, nbytes
    monkeypatch.setattr(M, "_chunk_workspace", filled)
    P.check_chunk(ops, "cpu", 1, T, Hqk, Hv, K, V, BF, backward=True, wrap=guarded, h0_std=0.1)
    assert len(parts) == 2   # the prep part, the state part: the gradients of the states are the last in it
    states = parts[1][-2 * Hv * K * V * 2:].view(BF).view(2, Hv, K * V)
    assert torch.isfinite(states).all()


@pytest.mark.parametrize("T,K,V", [(33, 64, 64), (70, 64, 192), (65, 128, 192)])
def test_kda_backward_where_the_sums_over_v_end(ops, T, K, V):
    """One pair of V blocks, R in two parts with the second cut short, waves without columns of K, a last chunk of one token."""
    P.check_kda(ops, "cpu", 1, T, 1, K, V, BF, backward=True, wrap=guarded, h0_std=0.1, seed=6)


def test_chunk_backward_without_initial_state(ops):
    P.check_chunk(ops, "cpu", 1, 70, 1, 1, 64, 64, F32, backward=True, with_h0=False, wrap=guarded)


@pytest.mark.parametrize("dtype,B,T,D,W,cu", [
    (F32, 2, 37, 16, 4, None), (BF, 1, 300, 32, 4, [0, 1, 3, 130, 131, 300]), (F32, 1, 9, 8, 3, [0, 2, 9]),
    (torch.float16, 2, 5, 8, 2, None), (F32, 3, 2, 8, 4, None), (F32, 1, 600, 8, 4, [0, 255, 257, 600]),
    (BF, 1, 41, 16, 4, list(range(42))), (F32, 9, 5, 8, 4, None),    # sequences shorter than a window or a tile
])
def test_conv1d(ops, dtype, B, T, D, W, cu):
    P.check_conv(ops, "cpu", B, T, D, W, dtype, cu=cu, residual=True, wrap=guarded)
    P.check_conv(ops, "cpu", B, T, D, W, dtype, cu=cu, bias=False, state=False, activation=None, wrap=guarded)


@pytest.mark.parametrize("T", [2, 100])
def test_conv1d_state_updated_in_place(ops, T):
    """The C entry with final_state = initial_state: the state is written by a launch of its own, behind the one whose
    first tiles read it."""
    B, D, W = 2, 16, 4
    gen = torch.Generator().manual_seed(0)
    x, w = torch.randn(B, T, D, generator=gen), torch.randn(W, D, generator=gen)
    h0 = torch.randn(B, D, W, generator=gen)
    want_y, want_fs = ops.causal_conv1d(x, w, initial_state=h0, output_final_state=True)
    y, lib = torch.empty_like(x), ops.lib
    lib.gdn_profile_enable(1)
    lib.check(lib.gdn_conv1d_fwd(ptr(x), ptr(w), None, None, ptr(h0), None, ptr(y), ptr(h0), B, T, B, D, W, 0, 0, None), "conv")
    launched = kernel_timings(lib)
    lib.gdn_profile_enable(0)
    assert torch.equal(y, want_y) and torch.equal(h0, want_fs)
    assert launched["conv1d_final_state_kernel"][1] == 1


@pytest.mark.parametrize("dtype,B,T,D,W", [(F32, 2, 1, 16, 4), (BF, 3, 5, 8, 4), (F32, 1, 3, 8, 2)])
def test_conv1d_update(ops, dtype, B, T, D, W):
    P.check_conv_update(ops, "cpu", B, T, D, W, dtype, wrap=guarded)


@pytest.mark.parametrize("dtype,shape,N,wdt", [
    (F32, (3, 5), 64, None), (BF, (70,), 128, None), (BF, (2, 9), 256, torch.float32), (F32, (33,), 16, None),
    (BF, (5,), 512, None), (F32, (4,), 256, None), (BF, (300,), 32, None),
])
def test_rms_norm_gated(ops, dtype, shape, N, wdt):
    P.check_rms_norm_gated(ops, "cpu", shape, N, dtype, weight_dtype=wdt, wrap=guarded)


@pytest.mark.parametrize("dtype,shape,N,wdt", [(F32, (3, 5), 64, None), (BF, (70,), 128, None), (BF, (2, 9), 128, torch.float32)])
def test_rms_norm_sigmoid_gated(ops, dtype, shape, N, wdt):
    P.check_rms_norm_gated(ops, "cpu", shape, N, dtype, weight_dtype=wdt, wrap=guarded, activation="sigmoid")


@pytest.mark.parametrize("activation", ["silu", "sigmoid"])
def test_rms_norm_far_gates(ops, activation):
    P.check_far_gates(ops, "cpu", activation)


@pytest.mark.parametrize("dtype,B,T,Hqk,Hv,K,V,l2,cu,pad", [
    (F32, 1, 100, 1, 2, 64, 64, True, None, 0),
    (BF, 2, 70, 2, 4, 128, 128, True, None, 0),
    (BF, 1, 140, 2, 2, 64, 64, False, [0, 5, 70, 71, 140], 16),
])
def test_chunk_on_unsplit_qkv(ops, dtype, B, T, Hqk, Hv, K, V, l2, cu, pad):
    P.check_chunk_qkv(ops, "cpu", B, T, Hqk, Hv, K, V, dtype, l2=l2, cu=cu, pad=pad, wrap=guarded, h0_std=0.1)


@pytest.mark.parametrize("dtype,B,T,Hqk,Hv,K,V,l2,cu,wdt,bwd", [
    (BF, 1, 100, 1, 2, 64, 128, True, None, None, True),
    (BF, 1, 140, 2, 2, 128, 64, False, [0, 5, 70, 71, 140], torch.float32, True),
    (F32, 1, 70, 1, 1, 64, 64, True, None, None, True),
    (BF, 2, 64, 1, 2, 64, 128, True, None, None, False),
])
def test_chunk_with_fused_norm(ops, dtype, B, T, Hqk, Hv, K, V, l2, cu, wdt, bwd):
    P.check_chunk_norm(ops, "cpu", B, T, Hqk, Hv, K, V, dtype, l2=l2, cu=cu, weight_dtype=wdt, backward=bwd,
                       wrap=guarded, h0_std=0.1)


@pytest.mark.parametrize("dtype,B,T,Hqk,Hv,K,V,l2,cu,bwd", [
    (BF, 1, 100, 1, 2, 64, 128, True, None, True),
    (BF, 1, 140, 2, 4, 64, 64, False, [0, 5, 70, 71, 140], False),
])
def test_chunk_on_unsplit_qkv_with_fused_norm(ops, dtype, B, T, Hqk, Hv, K, V, l2, cu, bwd):
    P.check_chunk_qkv_norm(ops, "cpu", B, T, Hqk, Hv, K, V, dtype, l2=l2, cu=cu, backward=bwd, wrap=guarded, h0_std=0.1)


@pytest.mark.parametrize("dtype,shape,Hv,pdt", [
    (F32, (2, 37), 6, None), (BF, (1, 300), 32, None), (BF, (3, 5), 48, torch.float32), (F32, (1,), 256, None),
    (BF, (1100,), 4, None),
])
def test_gdn_gates(ops, dtype, shape, Hv, pdt):
    P.check_gdn_gates(ops, "cpu", shape, Hv, dtype, param_dtype=pdt, wrap=guarded)


@pytest.mark.parametrize("dtype,B,steps,Hqk,Hv,K,V,W,pdt", [
    (F32, 2, 3, 1, 2, 64, 64, 4, None), (BF, 2, 4, 2, 4, 128, 128, 4, None), (BF, 1, 2, 1, 2, 64, 128, 3, torch.float32),
])
def test_decode_step(ops, dtype, B, steps, Hqk, Hv, K, V, W, pdt):
    P.check_decode_step(ops, "cpu", B, steps, Hqk, Hv, K, V, W, dtype, param_dtype=pdt, wrap=guarded)


@pytest.mark.parametrize("dtype,B,steps,Hqk,Hv,V,pdt,whole", [
    (BF, 2, 2, 1, 1, 64, None, True), (F32, 2, 2, 2, 2, 64, None, True), (F32, 1, 2, 1, 1, 128, None, True),
    (BF, 3, 2, 2, 4, 64, None, True), (BF, 3, 2, 1, 4, 64, torch.float32, True), (BF, 2, 2, 1, 2, 128, None, True),
    (BF, 1, 1, 1, 8, 64, None, False), (BF, 2, 2, 1, 4, 128, None, True), (BF, 1, 1, 1, 3, 64, None, False),
    (BF, 1, 1, 1, 3, 128, None, False), (F32, 1, 1, 1, 8, 128, None, False),
])
def test_decode_step_in_one_launch(ops, dtype, B, steps, Hqk, Hv, V, pdt, whole):
    """1, 2 and 4 slabs of 64 columns to a workgroup, 4 of 128 in place of 8; 3 of either and 8 of 128 take the two launches."""
    P.check_decode_step(ops, "cpu", B, steps, Hqk, Hv, 128, V, 4, dtype, param_dtype=pdt, wrap=guarded, one_launch=whole)


@pytest.mark.parametrize("dtype,T,W,cu", [(BF, 5, 4, [0, 3]), (F32, 64, 3, [0, 0, 2, 7]), (BF, 40, 8, [0, 17, 17]), (F32, 7, 1, [0, 5])])
def test_conv1d_rows_behind_the_last_sequence(ops, dtype, T, W, cu):
    P.check_conv_padded_rows(ops, "cpu", T, W, dtype, cu, wrap=guarded)


@pytest.mark.parametrize("dtype,V", [(BF, 64), (F32, 128)])
def test_decode_step_without_a_state(ops, dtype, V):
    P.check_decode_step_without_state(ops, "cpu", 2, 1, 1, 128, V, dtype, wrap=guarded)


@pytest.mark.parametrize("dtype,B,T,D,W,S", [(F32, 2, 3, 16, 4, 6), (BF, 2, 2, 8, 3, 3), (BF, 1, 1, 8, 4, 3)])
def test_conv1d_update_general_state_length(ops, dtype, B, T, D, W, S):
    P.check_conv_update(ops, "cpu", B, T, D, W, dtype, S=S, wrap=guarded)


def _random_case(seed):
    import random
    rng = random.Random(seed)
    B = rng.choice([1, 1, 2])
    T = rng.randint(1, 200)
    Hqk = rng.choice([1, 2])
    Hv = Hqk * rng.choice([1, 2, 4])
    K, V = rng.choice([64, 128]), rng.choice([64, 128, 192])
    cu = None
    if B == 1 and rng.random() < 0.6:
        cuts = sorted(rng.sample(range(0, T + 1), min(T + 1, rng.randint(0, 4))))
        cu = [0] + cuts + [T]
    return (BF if seed % 2 else F32), B, T, Hqk, Hv, K, V, rng.random() < 0.7, cu


def _one_output_gradients(ops, device, kda):
    """A loss that uses only one of the two outputs reaches the backward pass with the other gradient undefined (the
    functions ask autograd not to fill it with zeros): the gradients from o alone and from the final state alone add up
    to those of the loss over both (linearity), in fp32."""
    import tests.parity as P
    B, T, H, K, V = 1, 130, 2, 64, 128
    if kda:
        x = P.kda_inputs(B, T, H, K, V, torch.float32, seed=7)
        names = ("q", "k", "v", "g", "beta", "h0", "A_log", "dt_bias")
    else:
        x = P.gdn_inputs(B, T, H, 2 * H, K, V, torch.float32, seed=7)
        names = ("q", "k", "v", "g", "beta", "h0")
    d = {n: t.to(device) for n, t in x.items()}

    def grads(use_o, use_ht):
        leaves = {n: d[n].clone().requires_grad_(True) for n in names}
        if kda:
            o, ht = ops.chunk_kda(leaves["q"], leaves["k"], leaves["v"], leaves["g"], leaves["beta"],
                                  initial_state=leaves["h0"], output_final_state=True, use_qk_l2norm_in_kernel=True,
                                  use_gate_in_kernel=True, use_beta_sigmoid_in_kernel=True, A_log=leaves["A_log"],
                                  dt_bias=leaves["dt_bias"])
        else:
            o, ht = ops.chunk_gated_delta_rule(leaves["q"], leaves["k"], leaves["v"], leaves["g"], leaves["beta"],
                                               initial_state=leaves["h0"], output_final_state=True,
                                               use_qk_l2norm_in_kernel=True)
        loss = 0
        if use_o:
            loss = loss + (o * d["do"]).sum()
        if use_ht:
            loss = loss + (ht * d["dht"]).sum()
        return torch.autograd.grad(loss, list(leaves.values()))
    both, only_o, only_ht = grads(True, True), grads(True, False), grads(False, True)
    for n, a, b, c in zip(names, both, only_o, only_ht):
        scale = max(a.abs().max().item(), 1e-6)
        assert ((b + c) - a).abs().max().item() <= 2e-5 * scale + 1e-6, n
        if n in ("k", "v", "h0"):   # the final state does not depend on q
            assert c.abs().max().item() > 0, n
        if n == "q":
            assert c.abs().max().item() == 0


@pytest.mark.parametrize("kda", [False, True])
def test_gradient_from_one_output_only(ops, kda):
    _one_output_gradients(ops, "cpu", kda)


@pytest.mark.parametrize("seed", range(8))
def test_chunk_random_shapes(ops, seed):
    """Seeded random shapes: ragged lengths, packed sequences with empty and one-token members, grouped heads."""
    dtype, B, T, Hqk, Hv, K, V, l2, cu = _random_case(seed)
    P.check_chunk(ops, "cpu", B, T, Hqk, Hv, K, V, dtype, l2=l2, cu=cu, backward=True, wrap=guarded, h0_std=0.1, seed=seed)


@pytest.mark.parametrize("dtype,B,T,Hqk,Hv,K,V,cu", [
    (BF, 1, 70, 1, 2, 64, 64, None),               # last chunk of 6 tokens: its second 32-row half does not exist
    (BF, 1, 200, 2, 4, 128, 128, None),
    (F32, 1, 97, 1, 2, 64, 64, [0, 33, 97]),
])
def test_chunk_backward_stays_inside_its_outputs(ops, dtype, B, T, Hqk, Hv, K, V, cu):
    """Grouped heads (later value heads add to the dq, dk rows of the first) with a short last chunk, outputs and
    workspace against guard pages: no kernel may touch rows past the end of dq, dk, dv."""
    P.check_chunk(ops, "cpu", B, T, Hqk, Hv, K, V, dtype, cu=cu, backward=True, wrap=guarded, h0_std=0.1)


def _random_conv_case(seed):
    import random
    rng = random.Random(1000 + seed)
    dtype = rng.choice([BF, F32, BF])
    B, T, W = rng.choice([1, 1, 2, 3]), rng.randint(1, 300), rng.randint(1, 8)
    D = rng.choice([8, 16, 64, 72, 256])
    cu = None
    if B == 1 and rng.random() < 0.6:
        cuts = sorted(rng.sample(range(0, T + 1), min(T + 1, rng.randint(0, 5))))
        cu = [0] + cuts + [T]
    return dict(B=B, T=T, D=D, W=W, dtype=dtype, cu=cu, residual=rng.random() < 0.5, bias=rng.random() < 0.7,
                state=rng.random() < 0.7, activation=rng.choice(["silu", None]), seed=seed)


@pytest.mark.parametrize("seed", range(6))
def test_conv1d_random_shapes(ops, seed):
    """Seeded random shapes of the convolution: widths 1..8, ragged and packed lengths, with and without bias,
    residual, initial state and activation."""
    c = _random_conv_case(seed)
    P.check_conv(ops, "cpu", c.pop("B"), c.pop("T"), c.pop("D"), c.pop("W"), c.pop("dtype"), wrap=guarded, **c)


@pytest.mark.parametrize("dtype,B,T,H,K,V,cu,kw", [
    (F32, 1, 64, 1, 64, 64, None, {}),
    (F32, 2, 100, 2, 128, 128, None, {}),
    (BF, 1, 200, 2, 128, 128, None, {}),
    (BF, 1, 140, 2, 64, 64, [0, 5, 70, 71, 140], dict(lower_bound=-5.0)),
    (F32, 1, 96, 1, 128, 192, [0, 1, 38, 96], dict(gate_in_kernel=False, beta_sigmoid=False, l2=False, transpose_state=False)),
    (BF, 1, 130, 1, 128, 64, None, dict(allow_neg=True, with_h0=False, g_dtype=torch.float32)),
])
def test_kda_forward(ops, dtype, B, T, H, K, V, cu, kw):
    P.check_kda(ops, "cpu", B, T, H, K, V, dtype, cu=cu, wrap=guarded, h0_std=0.1, **kw)


@pytest.mark.parametrize("dtype,B,T,H,K,V,cu,kw", [
    (F32, 1, 64, 1, 64, 64, None, {}),
    (F32, 1, 100, 2, 128, 128, None, {}),
    (BF, 1, 200, 2, 128, 128, None, {}),
    (BF, 1, 140, 2, 64, 64, [0, 5, 70, 71, 140], dict(lower_bound=-5.0)),
    (F32, 1, 96, 1, 128, 64, [0, 1, 38, 96], dict(gate_in_kernel=False, beta_sigmoid=False, l2=False, transpose_state=False)),
    (BF, 1, 130, 1, 128, 64, None, dict(allow_neg=True, with_h0=False, g_dtype=torch.float32)),
])
def test_kda_backward(ops, dtype, B, T, H, K, V, cu, kw):
    errs = P.check_kda(ops, "cpu", B, T, H, K, V, dtype, cu=cu, backward=True, wrap=guarded, h0_std=0.1, **kw)
    print({n: f"{e:.2e}" for n, e in errs.items()})


def _random_kda_case(seed):
    import random
    rng = random.Random(1000 + seed)
    B = rng.choice([1, 1, 2])
    T = rng.randint(1, 200)
    H = rng.choice([1, 2, 3])
    K, V = rng.choice([64, 128]), rng.choice([64, 128, 192])
    cu = None
    if B == 1 and rng.random() < 0.6:
        cuts = sorted(rng.sample(range(0, T + 1), min(T + 1, rng.randint(0, 4))))
        cu = [0] + cuts + [T]
    kw = dict(gate_in_kernel=rng.random() < 0.7, beta_sigmoid=rng.random() < 0.7, l2=rng.random() < 0.7,
              transpose_state=rng.random() < 0.5, with_h0=rng.random() < 0.7, allow_neg=rng.random() < 0.3)
    if kw["gate_in_kernel"] and rng.random() < 0.4:
        kw["lower_bound"] = -5.0
    if not kw["beta_sigmoid"]:
        kw["allow_neg"] = False   # the doubled beta is an option of the in-kernel sigmoid
    return (BF if seed % 2 else F32), B, T, H, K, V, cu, kw


@pytest.mark.parametrize("seed", range(4))
def test_kda_random_shapes(ops, seed):
    """Seeded random shapes and options of chunk_kda, forward and backward: ragged and packed lengths with empty
    members, both state layouts, with and without the in-kernel gate, sigmoid and norm."""
    dtype, B, T, H, K, V, cu, kw = _random_kda_case(seed)
    P.check_kda(ops, "cpu", B, T, H, K, V, dtype, cu=cu, backward=True, wrap=guarded, h0_std=0.1, seed=seed, **kw)


@pytest.mark.parametrize("dtype,B,T,H,K,V,cu,kw", [
    (F32, 2, 100, 2, 128, 64, None, {}),
    (BF, 1, 200, 2, 64, 128, [0, 70, 70, 200], dict(transpose_state=False)),
    (BF, 1, 130, 1, 128, 128, None, dict(with_h0=False)),
])
def test_kda_intermediate_states(ops, dtype, B, T, H, K, V, cu, kw):
    """The states at chunk entries, written out from the workspace's tiles in both layouts."""
    errs = P.check_kda(ops, "cpu", B, T, H, K, V, dtype, cu=cu, wrap=guarded, h0_std=0.1, states=True, **kw)
    assert "h" in errs


@pytest.fixture(scope="module")
def ops256():
    """A device of 256 compute units: few heads and 64 chunks a sequence make the recurrences run cut into segments."""
    return emu_ops(256)


@pytest.mark.parametrize("kda", [False, True])
def test_cut_launch_hands_the_state_of_an_empty_sequence_through(ops256, kda):
    """An empty sequence beside a long one: its final state is its initial state and its initial state's gradient the final
    state's, bit for bit, infinities and NaN included."""
    T = 8193
    x = (P.kda_inputs(1, T, 1, 128, 128, BF, N=2) if kda else P.gdn_inputs(1, T, 1, 1, 128, 128, BF, N=2))
    h0, dht = x["h0"].clone(), torch.randn(x["h0"].shape, generator=torch.Generator().manual_seed(1))
    h0[0, 0, 3, 5], h0[0, 0, 7, 9], dht[0, 0, 2, 11] = float("inf"), float("nan"), -float("inf")
    leaf = {n: guarded(x[n]).requires_grad_(True) for n in ("q", "k", "v", "g", "beta")}
    h0 = guarded(h0).requires_grad_(True)
    kw = dict(initial_state=h0, output_final_state=True, use_qk_l2norm_in_kernel=True,
              cu_seqlens=torch.tensor([0, 0, T], dtype=torch.int64))
    if kda:
        o, ht = ops256.chunk_kda(*leaf.values(), use_gate_in_kernel=True, use_beta_sigmoid_in_kernel=True,
                                 A_log=guarded(x["A_log"]), dt_bias=guarded(x["dt_bias"]), **kw)
    else:
        o, ht = ops256.chunk_gated_delta_rule(*leaf.values(), **kw)
    dh0, = torch.autograd.grad([o, ht], [h0], [torch.ones_like(o), dht])
    assert torch.equal(ht[0].view(torch.int32), h0[0].view(torch.int32))
    assert torch.equal(dh0[0].view(torch.int32), dht[0].view(torch.int32))
    assert ht[1].isfinite().all() and dh0[1].isfinite().all()


@pytest.mark.parametrize("kda", [False, True])
def test_cut_launch_carries_a_slowly_decaying_state(ops, ops256, kda):
    """The maps, the chain and the cut recurrences against guard pages, and against the uncut recurrences."""
    P.check_cut_against_uncut(ops256, "cpu", 4097, 1, 1, kda, uncut_ops=ops, wrap=guarded)
