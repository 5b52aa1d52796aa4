"""GPU parity where the host picks another kernel or another split: shapes on both sides of each line, and the
smallest and largest of what each variant takes, against the oracle.

Tolerances are those of the dedicated tests and follow from the types: an fp32 state or tape is held to 1e-4 (a few
hundred roundings of 6e-8), bf16/f16 outputs to 2e-2 (the rounding of weights, partial rows and output)."""

import math

import numpy as np
import pytest
import torch

from oracle import dflash_oracle as O

pytestmark = pytest.mark.gpu


def host(t):
    return t.detach().float().cpu().numpy()


def dev(a, dt=torch.float32):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda", dt)


# step-by-step GatedDelta kernel: lanes per state row (16, 32 or 64) by B*Hv*Dv against 256 compute units
@pytest.mark.parametrize("Dk,Hv,Dv", [(128, 16, 128), (128, 17, 128), (256, 8, 128), (256, 9, 128), (256, 16, 128), (256, 17, 120)],
                         ids=lambda v: str(v))
@pytest.mark.parametrize("T", [1, 3, 4, 13, 17])
def test_step_kernel_lanes_per_row(gpu_lib, Dk, Hv, Dv, T):
    from swiftlm_amd import DFlashKernels as K

    d = O.make_gdn_inputs(Dk + Hv + T, 1, T, 1, Hv, Dk, Dv, in_dtype="bf16", vec_gate=True)
    mask = np.ones((1, T), np.float32)
    mask[0, T // 2] = float(T == 1)
    y, s, tape = K.gated_delta_kernel_with_tape(*[dev(d[n], torch.bfloat16) for n in ("q", "k", "v", "g", "beta")], dev(d["state"]), dev(mask))
    yw, sw, tw = O.gated_delta_ops_with_tape(d["q"], d["k"], d["v"], d["g"], d["beta"], d["state"], mask, dtype=np.float64)
    np.testing.assert_allclose(host(s), sw, rtol=1e-4, atol=1e-6)
    np.testing.assert_allclose(host(tape), tw, rtol=1e-4, atol=1e-5)
    np.testing.assert_allclose(host(y), yw, rtol=2e-2, atol=2e-2)


# ... and outputs written through where a compute unit has a second workgroup (fp32 state): as many workgroups as compute units, and a head more
@pytest.mark.parametrize("Dk,tiles", [(128, 8), (64, 4), (256, 8), (96, 4)], ids=str)
@pytest.mark.parametrize("more", [0, 1])
@pytest.mark.parametrize("masked", [False, True])
def test_step_kernel_stores(gpu_lib, Dk, tiles, more, masked):
    from swiftlm_amd import DFlashKernels as K

    rows = 32 if Dk == 96 else 16                      # of a workgroup
    T, Hv, Dv = 5, torch.cuda.get_device_properties(0).multi_processor_count // tiles + more, rows * tiles
    d = O.make_gdn_inputs(Dk + Hv, 1, T, 1, Hv, Dk, Dv, in_dtype="bf16", vec_gate=True)
    mask = np.ones((1, T), np.float32) if masked else None
    if masked:
        mask[0, 2] = 0
    y, s, tape = K.gated_delta_kernel_with_tape(*[dev(d[n], torch.bfloat16) for n in ("q", "k", "v", "g", "beta")], dev(d["state"]),
                                                None if mask is None else dev(mask))
    yw, sw, tw = O.gated_delta_ops_with_tape(d["q"], d["k"], d["v"], d["g"], d["beta"], d["state"], mask, dtype=np.float64)
    np.testing.assert_allclose(host(s), sw, rtol=1e-4, atol=1e-6)
    np.testing.assert_allclose(host(tape), tw, rtol=1e-4, atol=1e-5)
    np.testing.assert_allclose(host(y), yw, rtol=2e-2, atol=2e-2)


# Tape replay of one layer, whose state is written through where every compute unit has a workgroup, or Dk is above 64: both sides; nothing beside it
@pytest.mark.parametrize("Dk,Dv", [(64, 64), (32, 128), (128, 32)], ids=str)
@pytest.mark.parametrize("less", [0, 1])
@pytest.mark.parametrize("state", ["f32", "bf16"])
def test_replay_stores(gpu_lib, Dk, Dv, less, state):
    from swiftlm_amd import DFlashKernels as K

    T, Hv = 5, torch.cuda.get_device_properties(0).multi_processor_count // 4 - less           # four workgroups a head
    sdt = {"f32": torch.float32, "bf16": torch.bfloat16}[state]
    d = O.make_gdn_inputs(Dk + Hv, 1, T, 1, Hv, Dk, Dv, in_dtype="bf16")
    tape = np.random.default_rng(Hv).standard_normal((1, T, Hv, Dv)).astype(np.float32)
    k, g, s0 = dev(d["k"], torch.bfloat16), dev(d["g"], torch.bfloat16), dev(O.quantize(d["state"], state), sdt)
    got = K.tape_replay_kernel(dev(tape), k, g, s0, None)
    want = O.tape_replay_ops(tape, d["k"], d["g"], host(s0), dtype=np.float64, requant=None if state == "f32" else state)
    # (bf16: rounded after every step; a sum of the other side of a tie is 2^-8 away, and five steps carry it on)
    tol = dict(rtol=1e-4, atol=1e-6) if state == "f32" else dict(rtol=2e-2, atol=2e-2)
    np.testing.assert_allclose(host(got), want, **tol)
    # the replay of two layers writes plainly: the same bits
    outs = [torch.empty_like(s0) for _ in range(2)]
    K.tape_replay_batched([dev(tape)] * 2, [k] * 2, [g] * 2, [s0, s0.clone()], outs, T)
    assert torch.equal(outs[0], got) and torch.equal(outs[1], got)


# ... and rows per thread: two where the one-row form takes several rounds (Dv beyond a whole tile of either)
@pytest.mark.parametrize("Dk,Hv,Dv,vec", [(128, 65, 128, True), (128, 98, 120, False), (256, 33, 128, True), (256, 98, 120, False)], ids=lambda v: str(v))
@pytest.mark.parametrize("T", [1, 2, 5, 16, 18])
@pytest.mark.parametrize("state", ["f32", "bf16"])
def test_step_kernel_rows_per_thread(gpu_lib, Dk, Hv, Dv, vec, T, state):
    from swiftlm_amd import DFlashKernels as K

    if state == "f32" and not vec:
        Dv -= 1                                        # (a whole number of tiles takes the chunked kernels)
    d = O.make_gdn_inputs(Dk + Hv + T, 1, T, 1, Hv, Dk, Dv, in_dtype="bf16", vec_gate=vec)
    d["state"] = O.quantize(d["state"], state)
    mask = np.ones((1, T), np.float32)
    mask[0, T // 2] = float(T == 1)
    sdt = {"f32": torch.float32, "bf16": torch.bfloat16}[state]
    # two copies of the batch: B * Hv * Dv beyond the line
    run = lambda x: torch.cat([x, x])
    y, s, tape = K.gated_delta_kernel_with_tape(*[run(dev(d[n], torch.bfloat16)) for n in ("q", "k", "v", "g", "beta")], run(dev(d["state"], sdt)), run(dev(mask)))
    assert torch.equal(y[0], y[1]) and torch.equal(s[0], s[1]) and torch.equal(tape[0], tape[1])
    if state == "f32":
        yw, sw, tw = O.gated_delta_ops_with_tape(d["q"], d["k"], d["v"], d["g"], d["beta"], d["state"], mask, dtype=np.float64)
        np.testing.assert_allclose(host(s[:1]), sw, rtol=1e-4, atol=1e-6)
        np.testing.assert_allclose(host(tape[:1]), tw, rtol=1e-4, atol=1e-5)
    else:
        yw, sw, tw = O.gated_delta_ops_with_tape(d["q"], d["k"], d["v"], d["g"], d["beta"], d["state"], mask, requant="bf16")
        np.testing.assert_allclose(host(s[:1]), sw, rtol=2e-2, atol=2e-2)
        np.testing.assert_allclose(host(tape[:1]), tw, rtol=2e-2, atol=2e-2)
    np.testing.assert_allclose(host(y[:1]), yw, rtol=2e-2, atol=2e-2)


# GatedDelta forward over more than one chunk of 16 steps: 2 to 9 chunks (the producer waves take every fourth), whole and ragged
# last chunks, one and several row tiles
@pytest.mark.parametrize("Dk,Dv", [(64, 16), (128, 128), (256, 32)], ids=lambda v: str(v))
@pytest.mark.parametrize("T", [17, 32, 33, 48, 63, 65, 80, 97, 131])
@pytest.mark.parametrize("masked", [False, True])
def test_long_forward(gpu_lib, Dk, Dv, T, masked):
    from swiftlm_amd import DFlashKernels as K

    d = O.make_gdn_inputs(Dk + T, 2, T, 2, 4, Dk, Dv, in_dtype="bf16")
    mask = None
    if masked:
        mask = np.ones((2, T), np.float32)
        mask[0, 15:18] = 0
        mask[1, T - 5:] = 0
    ins = [dev(d[n], torch.bfloat16) for n in ("q", "k", "v", "g", "beta")]
    dmask = None if mask is None else dev(mask)
    y, s, tape = K.gated_delta_kernel_with_tape(*ins, dev(d["state"]), dmask)
    yw, sw, tw = O.gated_delta_ops_with_tape(d["q"], d["k"], d["v"], d["g"], d["beta"], d["state"], mask, dtype=np.float64)
    np.testing.assert_allclose(host(s), sw, rtol=1e-4, atol=1e-6)
    np.testing.assert_allclose(host(tape), tw, rtol=1e-4, atol=1e-5)
    np.testing.assert_allclose(host(y), yw, rtol=2e-2, atol=2e-2)
    # the same rows 8 bytes off a 16-byte line take the chunk-by-chunk kernel: the same sums in another order
    off = [torch.empty(t.numel() + 4, dtype=t.dtype, device="cuda")[4:].view(t.shape).copy_(t) if i < 2 else t for i, t in enumerate(ins)]
    y2, s2, tape2 = K.gated_delta_kernel_with_tape(*off, dev(d["state"]), dmask)
    np.testing.assert_allclose(host(s2), host(s), rtol=1e-4, atol=1e-6)
    np.testing.assert_allclose(host(tape2), host(tape), rtol=1e-4, atol=1e-5)
    np.testing.assert_allclose(host(y2), host(y), rtol=2e-2, atol=2e-2)


# A mask of any type, its elements around the line (0.5 does not run, the next value above does, NaN does not): the bits of zeros and ones.
# Chunks whose mask is asked for ahead of the loop (the first four), in it, and in a ragged last one; two sequences; any address.
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16, torch.uint8], ids=str)
@pytest.mark.parametrize("Dk,T", [(64, 17), (128, 70), (128, 131), (256, 97)])
def test_long_forward_mask_types(gpu_lib, Dk, T, dt):
    from swiftlm_amd import DFlashKernels as K

    d = O.make_gdn_inputs(Dk + T, 2, T, 2, 4, Dk, 32, in_dtype="bf16")
    ins = [dev(d[n], torch.bfloat16) for n in ("q", "k", "v", "g", "beta")]
    if dt == torch.uint8:
        values, on = [0, 1, 2, 255], [0, 1, 1, 1]
    else:
        above = float(torch.tensor(0.5, dtype=dt).float()) * (1 + torch.finfo(dt).eps)
        values, on = [0.0, 0.5, above, 1.0, float("nan"), float("inf"), -1.0, torch.finfo(dt).tiny], [0, 0, 1, 1, 0, 1, 0, 0]
    pick = np.random.default_rng(T).integers(0, len(values), (2, T))
    mask = torch.empty(2 * T + 1, dtype=dt, device="cuda")[1:].view(2, T).copy_(torch.tensor(values, dtype=torch.float64).to(dt)[torch.from_numpy(pick)])
    plain = np.array(on, np.float32)[pick]
    want = K.gated_delta_kernel_with_tape(*ins, dev(d["state"]), dev(plain))
    for got, w in zip(K.gated_delta_kernel_with_tape(*ins, dev(d["state"]), mask), want):
        assert torch.equal(got, w)
    sw = O.gated_delta_ops_with_tape(d["q"], d["k"], d["v"], d["g"], d["beta"], d["state"], plain, dtype=np.float64)[1]
    np.testing.assert_allclose(host(want[1]), sw, rtol=1e-4, atol=1e-6)


# v, y and the tape may lie at any address of their elements: the kernel of aligned ones, hence its bits, and nothing beside them
@pytest.mark.parametrize("off", [1, 2, 4])
def test_long_forward_v_alignment(gpu_lib, off):
    from swiftlm_amd import DFlashKernels as K
    from swiftlm_amd._lib import native

    d = O.make_gdn_inputs(3, 1, 50, 2, 4, 128, 48, in_dtype="bf16")
    q, k, v, g, beta = [dev(d[n], torch.bfloat16) for n in ("q", "k", "v", "g", "beta")]
    moved = torch.empty(v.numel() + off, dtype=v.dtype, device="cuda")[off:].view(v.shape).copy_(v)
    y, s, tape = K.gated_delta_kernel_with_tape(q, k, moved, g, beta, dev(d["state"]))
    for got, want in zip((y, s, tape), K.gated_delta_kernel_with_tape(q, k, v, g, beta, dev(d["state"]))):
        assert torch.equal(got, want)
    ym, tm = (torch.full((t.numel() + 2 * off,), 7.0, dtype=t.dtype, device="cuda") for t in (y, tape))
    inner = lambda t, like: t[off:-off].view(like.shape)
    sm = torch.empty_like(s)
    native.gated_delta_into(native.current_stream(), q, k, moved, g, beta, dev(d["state"]), sm, inner(ym, y), inner(tm, tape), 2, 4, 128, 48)
    assert torch.equal(inner(ym, y), y) and torch.equal(inner(tm, tape), tape) and torch.equal(sm, s)
    assert all(bool((t[:off] == 7).all() and (t[-off:] == 7).all()) for t in (ym, tm))
    yw, sw, tw = O.gated_delta_ops_with_tape(d["q"], d["k"], d["v"], d["g"], d["beta"], d["state"], dtype=np.float64)
    np.testing.assert_allclose(host(s), sw, rtol=1e-4, atol=1e-6)
    np.testing.assert_allclose(host(tape), tw, rtol=1e-4, atol=1e-5)
    np.testing.assert_allclose(host(y), yw, rtol=2e-2, atol=2e-2)


# A value that is not finite stays in its row and in the steps from it on; a chunk whose solve matrix overflows (1e4^15) where no
# delta does has the deltas that substitution gives.
def test_long_forward_not_finite(gpu_lib):
    from swiftlm_amd import DFlashKernels as K

    T, row, step = 50, 5, 23
    d = O.make_gdn_inputs(1, 1, T, 2, 4, 128, 32, in_dtype="bf16")
    q, k, v, g, beta = [dev(d[n], torch.bfloat16) for n in ("q", "k", "v", "g", "beta")]
    y, s, tape = K.gated_delta_kernel_with_tape(q, k, v, g, beta, dev(d["state"]))
    for bad in (float("inf"), float("nan")):
        vb = v.clone()
        vb[0, step, 1, row] = bad
        yb, sb, tb = K.gated_delta_kernel_with_tape(q, k, vb, g, beta, dev(d["state"]))
        np.testing.assert_allclose(host(tb[:, :step]), host(tape[:, :step]), rtol=1e-4, atol=1e-5)
        assert not torch.isfinite(tb[0, step:, 1, row]).any() and not torch.isfinite(sb[0, 1, row]).any()
        keep = torch.ones_like(tape, dtype=torch.bool)
        keep[0, :, 1, row] = False
        np.testing.assert_allclose(host(tb[keep]), host(tape[keep]), rtol=1e-4, atol=1e-5)
        keep[0, :step, 1, row] = True
        np.testing.assert_allclose(host(yb[keep]), host(y[keep]), rtol=2e-2, atol=2e-2)
    big = torch.full_like(k, 10.0)                            # k.k = 12800
    y, s, tape = K.gated_delta_kernel_with_tape(q, big, torch.zeros_like(v), torch.ones_like(g), torch.ones_like(beta), torch.zeros_like(s))
    assert not y.any() and not s.any() and not tape.any()


# ... and y of the steps in front of it is what it is without it, in every form of the forward: one chunk, chunk by chunk (f16, fp32),
# several chunks, and with a decay per channel the steps one by one and 16 at a time.  Whatever holds it: v, which one state row
# sees, or k, q, the gate or beta.
@pytest.mark.parametrize("vec", [False, True], ids=["head", "channel"])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("T,step", [(16, 0), (16, 5), (13, 12), (50, 23), (50, 49)], ids=str)
def test_forward_not_finite_is_causal(gpu_lib, T, step, dt, vec):
    from swiftlm_amd import DFlashKernels as K

    d = O.make_gdn_inputs(T + step, 1, T, 2, 4, 128, 32, in_dtype="bf16", vec_gate=vec)
    ins = {n: dev(d[n], dt) for n in ("q", "k", "v", "g", "beta")}
    state = dev(d["state"])
    y, s, tape = K.gated_delta_kernel_with_tape(*ins.values(), state)
    for name in ins:
        for bad in (float("inf"), float("nan")):
            with_bad = {n: x.clone() for n, x in ins.items()}
            x = with_bad[name][0, step, 0]
            x[...] = bad
            yb, sb, tb = K.gated_delta_kernel_with_tape(*with_bad.values(), state)
            np.testing.assert_allclose(host(yb[:, :step]), host(y[:, :step]), rtol=2e-2, atol=2e-2, err_msg=f"{bad} in {name}")
            np.testing.assert_allclose(host(tb[:, :step]), host(tape[:, :step]), rtol=1e-4, atol=1e-5, err_msg=f"{bad} in {name}")
            assert not torch.isfinite(yb[0, step, 0]).any()
            for h in (2, 3):                                  # heads of the other key head
                np.testing.assert_allclose(host(yb[:, :, h]), host(y[:, :, h]), rtol=2e-2, atol=2e-2, err_msg=f"{bad} in {name}")
                np.testing.assert_allclose(host(sb[:, h]), host(s[:, h]), rtol=1e-4, atol=1e-6, err_msg=f"{bad} in {name}")


# A masked step keeps the state and writes zeros, whatever its rows hold (padding): every form of the forward, as above, and an fp16
# state, gives the bits that it gives over zeros there; a state row that is not finite makes no delta either.
@pytest.mark.parametrize("vec", [False, True], ids=["head", "channel"])
@pytest.mark.parametrize("dt,state", [("bf16", "f32"), ("f16", "f32"), ("f32", "f32"), ("f16", "f16")], ids=str)
@pytest.mark.parametrize("T,off", [(16, [0]), (16, [3, 4, 9]), (13, [12]), (50, [0, 15, 16]), (50, [23, 48, 49])], ids=str)
def test_masked_steps_hold_anything(gpu_lib, T, off, dt, state, vec):
    from swiftlm_amd import DFlashKernels as K

    types = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
    d = O.make_gdn_inputs(T + len(off), 1, T, 2, 4, 128, 32, in_dtype="bf16", vec_gate=vec)
    d["state"] = O.quantize(d["state"], state)
    mask = np.ones((1, T), np.float32)
    mask[0, off] = 0
    ins = {n: dev(d[n], types[dt]) for n in ("q", "k", "v", "g", "beta")}
    for x in ins.values():
        x[0, off] = 0
    s0 = dev(d["state"], types[state])
    run = lambda x, s: K.gated_delta_kernel_with_tape(*x.values(), s, dev(mask))
    y, s, tape = run(ins, s0)
    if state == "f32":
        yw, sw, tw = O.gated_delta_ops_with_tape(d["q"], d["k"], d["v"], d["g"], d["beta"], d["state"], mask, dtype=np.float64)
        np.testing.assert_allclose(host(s), sw, rtol=1e-4, atol=1e-6)
        np.testing.assert_allclose(host(tape), tw, rtol=1e-4, atol=1e-5)
        np.testing.assert_allclose(host(y), yw, rtol=2e-2, atol=2e-2)
    for name in ins:
        for bad in (float("inf"), float("nan")):
            held = {n: x.clone() for n, x in ins.items()}
            held[name][0, off] = bad
            for got, want in zip(run(held, s0), (y, s, tape)):
                assert torch.equal(got, want), f"{bad} in {name}"
    for bad in (float("inf"), float("nan")):
        sb = s0.clone()
        sb[0, 1, 5, 7] = bad
        yb, _, tb = run(ins, sb)
        assert not tb[0, off].any() and not yb[0, off].any()
        first = min(t for t in range(T) if t not in off)
        assert not torch.isfinite(tb[0, first, 1, 5])


def attend(q, k, v, lens, D, **kw):
    from swiftlm_amd import DFlashKernels as K

    out, lse = K.batched_sdpa_2pass(q, k, v, 1.0 / math.sqrt(D), return_lse=True, **kw)
    torch.cuda.synchronize()
    for b, n in enumerate(lens):
        ow, lw = O.sdpa_block_causal(host(q[b:b + 1]), host(k[b:b + 1, :, :n]), host(v[b:b + 1, :, :n]), 1.0 / math.sqrt(D))
        np.testing.assert_allclose(host(out[b]), ow[0], rtol=2e-2, atol=2e-2, err_msg=f"sequence {b} of {n} keys")
        np.testing.assert_allclose(host(lse[b]), lw[0], rtol=2e-3, atol=2e-3, err_msg=f"sequence {b} of {n} keys")
    return out, lse


def tensors(seed, B, Hq, Hk, N, D, dt=torch.bfloat16):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn(B, h, n, D, generator=g, device="cuda").to(dt) for h, n in ((Hq, 16), (Hk, N), (Hk, N))]


# one split writes the output itself (up to four tiles of 32 keys); with few splits a wave merges a row, with more a workgroup
@pytest.mark.parametrize("N", [16, 17, 32, 33, 128, 129, 250, 1024, 1056, 2048, 2080])
@pytest.mark.parametrize("Hq,Hk,D", [(3, 1, 256), (4, 2, 128)])
def test_attention_split_counts(gpu_lib, N, Hq, Hk, D):
    attend(*tensors(N + D, 1, Hq, Hk, N, D), [N], D)


# a workgroup per row has as many partial rows in flight per thread as the splits ask for: 4, 8, 12, 16 (above up to 65 splits at D = 256)
@pytest.mark.parametrize("D,N,S", [(256, 3072, 96), (256, 3104, 97), (256, 4096, 128), (256, 40000, 209), (128, 2080, 65), (128, 4096, 128), (128, 5000, 157),
                                   (128, 33000, 172), (128, 65568, 256)])
def test_combine_rows_in_flight(gpu_lib, D, N, S):
    assert splits(1, 3, 1, N, D) == S
    attend(*tensors(N + D, 1, 3, 1, N, D), [N], D)


def first_launch(B, Hq, Hk, N, D):
    from swiftlm_amd import _lib

    shapes = (_lib.LaunchShape * 2)()
    assert _lib.load().dflash_profile_sdpa_launches(_lib.BF16, B, Hq, Hk, N, D, shapes) > 0
    return shapes[0]


def short_splits(B, Hq, Hk, N, D):
    """Splits of the form with a workgroup per query head, 0 where the form with shared tiles runs; by the library's own account."""
    shape = first_launch(B, Hq, Hk, N, D)
    return shape.grid_x // Hk if shape.kernel == b"sdpa_short_kernel" else 0


# Short contexts in one launch, up to a line of keys that depends on the query heads (B * Hq), then a few splits of the same form, then
# the form with shared tiles, which more heads than compute units take at once.  Tiles of 32 (D = 128) and 16 keys, eight waves, one
# tile a wave and more; the second sequence leaves splits without a tile; 24 heads whose splits are rounded to whole XCDs.
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("Hq,Hk,D,N,S", [
    (2, 1, 128, 31, 1), (3, 1, 128, 257, 1), (8, 1, 128, 896, 1), (8, 1, 128, 897, 16), (32, 8, 128, 1152, 1), (32, 8, 128, 1153, 4), (64, 8, 128, 1152, 1),
    (64, 8, 128, 1153, 0), (66, 6, 128, 1152, 1), (66, 6, 128, 1153, 0), (130, 2, 128, 100, 0),
    (2, 1, 256, 17, 1), (3, 1, 256, 129, 1), (8, 1, 256, 416, 1), (8, 1, 256, 417, 8), (16, 2, 256, 416, 1), (16, 2, 256, 417, 8), (32, 8, 256, 576, 1),
    (32, 8, 256, 577, 4), (64, 8, 256, 576, 1), (64, 8, 256, 577, 0), (66, 6, 256, 576, 1), (66, 6, 256, 577, 0), (130, 2, 256, 129, 0),
    (1, 1, 128, 2048, 16), (1, 1, 128, 2049, 0), (12, 2, 128, 3200, 8), (12, 2, 128, 3201, 0), (4, 1, 128, 3584, 16), (4, 1, 128, 3585, 0), (32, 8, 128, 1600, 4),
    (32, 8, 128, 1601, 0), (6, 2, 256, 5760, 20), (6, 2, 256, 5761, 0), (16, 8, 256, 2304, 8), (16, 8, 256, 2305, 0), (1, 1, 256, 9000, 64)])
def test_short_contexts(gpu_lib, Hq, Hk, D, N, S, dt):
    from swiftlm_amd import DFlashKernels as K

    assert short_splits(2, Hq, Hk, N, D) == S
    lens = [N, max(16, N // 2 + 1) if N < 4000 else 17]
    q, k, v = tensors(N + D, 2, Hq, Hk, N, D, dt)
    kv_len = torch.tensor(lens, dtype=torch.int32, device="cuda")
    out, lse = attend(q, k, v, lens, D, kv_len=kv_len)
    # masked and fused calls give the same bits
    zero = torch.zeros(2, Hq, 16, N, dtype=dt, device="cuda")
    masked = K.batched_sdpa_2pass(q, k, v, 1.0 / math.sqrt(D), zero, return_lse=True, kv_len=kv_len)
    new = [torch.stack([x[b, :, n - 16:n] for b, n in enumerate(lens)]).contiguous() for x in (k, v)]
    kc, vc = k.clone(), v.clone()
    for b, n in enumerate(lens):
        kc[b, :, n - 16:n], vc[b, :, n - 16:n] = float("nan"), float("nan")
    fused = K.batched_sdpa_2pass_append(q, kc, vc, *new, 1.0 / math.sqrt(D), N, cache_len=kv_len - 16, return_lse=True)
    for o, l in (masked, fused):
        assert torch.equal(o, out) and torch.equal(l, lse)
    assert torch.equal(kc, k) and torch.equal(vc, v)


# The few splits end at as many keys to a split where four and more query heads share a KV head: both sides of the line
@pytest.mark.parametrize("Hq,Hk,D,last,S", [(8, 2, 256, 4608, 16), (16, 2, 256, 2304, 8), (4, 1, 256, 9216, 32), (12, 2, 256, 2304, 8), (8, 1, 128, 3584, 16),
                                            (6, 1, 128, 3584, 16)], ids=str)
def test_few_splits_end_with_shared_kv_heads(gpu_lib, Hq, Hk, D, last, S):
    for N, want in ((last, S), (last + 1, 0)):
        assert short_splits(2, Hq, Hk, N, D) == want
        attend(*tensors(N + D, 2, Hq, Hk, N, D), [N, N], D)


# One split, with V's channels in four parts, two or one by how many heads the call has: a head's bits are the same, at contexts of one
# key, a tile, a tile and one more, a wave's second tile, and a mask that hides a tile from some rows.
@pytest.mark.parametrize("D,N", [(128, 17), (128, 64), (128, 257), (128, 300), (256, 16), (256, 65), (256, 129), (256, 400)])
def test_short_parts_same_bits(gpu_lib, D, N):
    from swiftlm_amd import DFlashKernels as K

    q, k, v = tensors(N + D, 5, 32, 4, N, D)
    mask = torch.zeros(5, 32, 16, N, dtype=q.dtype, device="cuda")
    mask[:, :, 3:5, :min(N - 16, 40)] = float("-inf")
    run = lambda n, m: K.batched_sdpa_2pass(q[:n], k[:n], v[:n], 1.0 / math.sqrt(D), None if m is None else m[:n], return_lse=True)
    assert [short_splits(n, 32, 4, N, D) for n in (2, 3, 5)] == [1, 1, 1]
    assert [first_launch(n, 32, 4, N, D).grid_y for n in (2, 3, 5)] == [8 * parts for parts in (4, 2, 1)]
    for m in (None, mask):
        few, some, many = run(2, m), run(3, m), run(5, m)
        for x, y, z in zip(few, some, many):
            assert torch.equal(x, z[:2]) and torch.equal(y, z[:3])
    attend(q[:2], k[:2], v[:2], [N, N], D)


# The mask's loads, four keys each in the form with shared tiles: rows of odd and even length, a last tile of one key and of all but
# one; one split of either form and several.
@pytest.mark.parametrize("N", [0, 1, 2, 3, 5, 31])
@pytest.mark.parametrize("Hq,Hk,D,base,short", [(3, 1, 256, 1184, True), (10, 2, 128, 1184, True), (64, 8, 256, 1184, False), (64, 8, 128, 1184, False),
                                                (130, 10, 128, 64, False), (130, 10, 256, 64, False)])
def test_mask_row_ends(gpu_lib, N, Hq, Hk, D, base, short):
    from swiftlm_amd import DFlashKernels as K

    N += base
    assert (short_splits(2, Hq, Hk, N, D) > 0) == short
    q, k, v = tensors(N + D, 2, Hq, Hk, N, D)
    g = torch.Generator(device="cuda").manual_seed(N)
    mask = torch.randn(2, Hq, 16, N, generator=g, device="cuda").masked_fill(torch.rand(2, Hq, 16, N, generator=g, device="cuda") < 0.3, float("-inf"))
    mask = mask.to(torch.bfloat16)
    out, lse = K.batched_sdpa_2pass(q, k, v, 1.0 / math.sqrt(D), mask, return_lse=True)
    ow, lw = O.sdpa_block_causal(host(q), host(k), host(v), 1.0 / math.sqrt(D), host(mask).astype(np.float64))
    np.testing.assert_allclose(host(out), ow, rtol=2e-2, atol=2e-2)
    np.testing.assert_allclose(host(lse), lw, rtol=2e-3, atol=2e-3)


# ragged batches of short sequences, every one with its own splits: one beside many, equal lengths, all at the minimum, 64 and 65
@pytest.mark.parametrize("lens", [[700, 16], [16, 17, 2000, 33], [500] * 5, [16] * 3 + [129], [40 + 3 * i for i in range(64)],
                                  [40 + 3 * i for i in range(65)]], ids=lambda v: f"{len(v)}x{max(v)}")
@pytest.mark.parametrize("D", [128, 256])
def test_ragged_short(gpu_lib, lens, D):
    assert not dealt(len(lens), 4, 2, max(lens), D)
    q, k, v = tensors(len(lens) + D, len(lens), 4, 2, max(lens), D)
    attend(q, k, v, lens, D, kv_len=torch.tensor(lens, dtype=torch.int32, device="cuda"))


# From a line on, in tiles of 32 keys per workgroup and with up to 64 sequences, a lane each, the workgroups are dealt by length.
def splits(B, Hq, Hk, N, D):
    from swiftlm_amd import DFlashKernels as K

    return K.sdpa_workspace_bytes(B, Hq, Hk, 16, N, D) // (B * Hq * 16 * (2 * D + 8))


def dealt(B, Hq, Hk, N, D, most=64):
    S = splits(B, Hq, Hk, N, D)
    fit = torch.cuda.get_device_properties(0).multi_processor_count // (Hk * -(-(Hq // Hk) // 8))
    W = min(fit, B * S)
    line = 6 if B * S > fit else 30 if W < 3 * B else 7 if D == 256 and W <= 8 * B and B <= 16 else 12
    return B <= most and W > B and (B - 1) * -(-N // 32) >= line * W


# Every form of the call, each with a sequence of more than 64 splits beside short ones: one wave merges a row at D = 128, a
# workgroup at D = 256.  Paged and fused calls give the bits of the dense one (the same shares, the same order).
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("D", [128, 256])
@pytest.mark.parametrize("lens", [[16384, 16, 17, 40], [33, 16384, 16383, 16], [9000, 8999, 16, 16382]], ids=str)
def test_ragged_shares_every_form(gpu_lib, lens, D, dt):
    from swiftlm_amd import DFlashKernels as K

    B, Hq, Hk, N, P, scale = 4, 4, 2, 16384, 64, 1.0 / math.sqrt(D)
    assert dealt(B, Hq, Hk, N, D) and splits(B, Hq, Hk, N, D) == 32
    q, k, v = tensors(sum(lens) + D, B, Hq, Hk, N, D, dt)
    n = torch.tensor(lens, dtype=torch.int32, device="cuda")
    out, lse = attend(q, k, v, lens, D, kv_len=n)
    mask = 0.1 * torch.randn(B, Hq, 16, N, generator=torch.Generator(device="cuda").manual_seed(N), device="cuda")
    mask[:, :, :, 32:64] = float("-inf")                      # a hidden tile among others, with values that are not finite
    mask = mask.to(dt)
    vm = v.clone()
    vm[:, :, 32:64] = float("nan")
    om, lm = K.batched_sdpa_2pass(q, k, vm, scale, mask, return_lse=True, kv_len=n)
    for b, m in enumerate(lens):
        want = O.sdpa_block_causal(host(q[b:b + 1]), host(k[b:b + 1, :, :m]), host(v[b:b + 1, :, :m]), scale, host(mask[b:b + 1, :, :, :m]).astype(np.float64))
        same_rows(om[b], lm[b], want[0][0], want[1][0])
    # fused append: the block's rows come from apart and end up in the cache
    kc, vc = k.clone(), v.clone()
    k_new, v_new = (torch.stack([t[b, :, m - 16:m] for b, m in enumerate(lens)]).contiguous() for t in (k, v))
    for b, m in enumerate(lens):
        kc[b, :, m - 16:m] = vc[b, :, m - 16:m] = 9.0
    oa, la = K.batched_sdpa_2pass_append(q, kc, vc, k_new, v_new, scale, N, cache_len=n - 16, return_lse=True)
    assert torch.equal(oa, out) and torch.equal(la, lse) and torch.equal(kc, k) and torch.equal(vc, v)
    # pages in any order
    order = torch.randperm(B * N // P, generator=torch.Generator().manual_seed(D))
    table = order.view(B, N // P).to(torch.int32).cuda()
    kp, vp = (torch.empty(B * N // P, Hk, P, D, dtype=dt, device="cuda") for _ in range(2))
    for pool, t in ((kp, k), (vp, v)):
        pool[order.cuda()] = t.view(B, Hk, N // P, P, D).transpose(1, 2).reshape(-1, Hk, P, D)
    op, lp = K.batched_sdpa_2pass_paged(q, kp, vp, table, scale, N, lengths=n, return_lse=True)
    assert torch.equal(op, out) and torch.equal(lp, lse)
    for b, m in enumerate(lens):
        for r in range(m - 16, m):
            kp[table[b, r // P], :, r % P] = vp[table[b, r // P], :, r % P] = 9.0
    op, lp = K.batched_sdpa_2pass_paged(q, kp, vp, table, scale, N, k_new=k_new, v_new=v_new, lengths=n - 16, return_lse=True)
    assert torch.equal(op, out) and torch.equal(lp, lse)
    for pool, t in ((kp, k), (vp, v)):
        assert torch.equal(pool[order.cuda()].view(B, N // P, Hk, P, D).transpose(1, 2).reshape(B, Hk, N, D), t)


# The combine kernels behind dealt splits: a wave with 4 or 16 rows in flight, a workgroup; as many sequences as a wave has lanes; a
# workgroup for every split, and fewer, as no more fit the chip at once.
@pytest.mark.parametrize("B,Hq,Hk,D,N,S", [(64, 2, 1, 128, 1600, 4), (64, 3, 1, 256, 1600, 4), (63, 1, 1, 128, 2000, 5), (16, 8, 1, 256, 6600, 16), (16, 2, 1, 256, 6600, 16), (11, 8, 1, 256, 6600, 24),
                                           (2, 1, 1, 128, 98304, 128), (2, 1, 1, 256, 98304, 128), (32, 8, 4, 128, 2000, 2),
                                           (3, 16, 2, 128, 16512, 43), (3, 4, 2, 256, 16000, 43), (5, 8, 8, 128, 2000, 7), (12, 8, 8, 256, 900, 3), (50, 8, 1, 128, 2000, 6)])
def test_ragged_shares_combine(gpu_lib, B, Hq, Hk, D, N, S):
    assert dealt(B, Hq, Hk, N, D) and splits(B, Hq, Hk, N, D) == S
    rng = np.random.default_rng(B + D)
    lens = [int(n) for n in np.exp(rng.uniform(math.log(16), math.log(N), B))]
    lens[B // 2] = N
    q, k, v = tensors(B + D, B, Hq, Hk, N, D)
    attend(q, k, v, lens, D, kv_len=torch.tensor(lens, dtype=torch.int32, device="cuda"))


def test_ragged_batch_of_more_sequences_than_lanes(gpu_lib):
    B, N, D = 65, 1600, 128
    assert not dealt(B, 2, 1, N, D) and dealt(B, 2, 1, N, D, most=B)
    lens = [16 + (N - 16) * i // (B - 1) for i in range(B)]
    q, k, v = tensors(B, B, 2, 1, N, D)
    attend(q, k, v, lens, D, kv_len=torch.tensor(lens, dtype=torch.int32, device="cuda"))


# the line: eight sequences of eight KV heads take four splits each
@pytest.mark.parametrize("D,N", [(256, 992), (256, 1024), (128, 1728), (128, 1760), (128, 2200)])
def test_ragged_shares_line(gpu_lib, D, N):
    import ctypes as C

    assert dealt(8, 8, 8, N, D) == (N not in (992, 1728))
    lens = [N, 16, N // 2, 17, 33, N, 700, 129]
    q, k, v = tensors(N + D, 8, 8, 8, N, D)
    status = torch.zeros(1, dtype=torch.int32, device="cuda")
    assert gpu_lib.dflash_set_status_word(C.c_void_p(status.data_ptr())) == 0
    try:
        given = torch.tensor(lens, dtype=torch.int32, device="cuda")
        attend(q, k, v, lens, D, kv_len=given)
        assert int(status) == 0
        given[5], given[1] = 9000, 3                # outside the bounds: flagged, and read as N and 16
        attend(q, k, v, lens, D, kv_len=given)
        assert int(status) == 1
    finally:
        assert gpu_lib.dflash_set_status_word(None) == 0


# (splits of its own; the test above has dealt ones)
def test_ragged_short_length_outside_the_bound_is_flagged_and_clamped(gpu_lib):
    import ctypes as C

    q, k, v = tensors(3, 3, 4, 2, 400, 128)
    status = torch.zeros(1, dtype=torch.int32, device="cuda")
    assert gpu_lib.dflash_set_status_word(C.c_void_p(status.data_ptr())) == 0
    try:
        attend(q, k, v, [400, 16, 200], 128, kv_len=torch.tensor([900, 3, 200], dtype=torch.int32, device="cuda"))
        assert int(status) == 1
    finally:
        assert gpu_lib.dflash_set_status_word(None) == 0


# A tile of 32 keys that a row sees nothing of leaves the row alone, whatever its V rows hold: in one split that writes the output
# itself and as the first, a middle and the last tile of a longer one.  Tolerances as above: the tile adds nothing to these rows.
def same_rows(out, lse, ow, lw):
    np.testing.assert_allclose(host(out), ow, rtol=2e-2, atol=2e-2)
    np.testing.assert_allclose(host(lse), lw, rtol=2e-3, atol=2e-3)


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("N", [33, 47, 97, 110, 129, 2049, 2063])
@pytest.mark.parametrize("Hq,Hk,D,short", [(3, 1, 256, True), (8, 8, 128, True), (264, 8, 128, False), (264, 8, 256, False)])
def test_last_tile_hidden_by_the_causal_rule(gpu_lib, N, Hq, Hk, D, short, bad):
    from swiftlm_amd import DFlashKernels as K

    assert (short_splits(1, Hq, Hk, N, D) > 0) == short
    q, k, v = tensors(N + D, 1, Hq, Hk, N, D)
    keys = N % 32                                             # of the last tile; row r sees keys up to N - 16 + r
    want = O.sdpa_block_causal(host(q), host(k), host(v), 0.1)
    v[:, :, N - keys:] = bad
    out, lse = K.batched_sdpa_2pass(q, k, v, 0.1, return_lse=True)
    same_rows(out[:, :, :16 - keys], lse[:, :, :16 - keys], want[0][:, :, :16 - keys], want[1][:, :, :16 - keys])
    assert not torch.isfinite(out[:, :, 15]).any()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("N,tiles", [(64, [1]), (100, [0, 2]), (128, [0]), (128, [1, 3]), (2048, [0]), (2048, [16, 33]), (2048, [48]), (2048, [0, 16, 47])],
                         ids=str)
@pytest.mark.parametrize("Hq,Hk,D,short", [(8, 8, 128, True), (32, 8, 256, True), (264, 8, 128, False), (264, 8, 256, False)])
def test_tiles_hidden_by_the_mask(gpu_lib, N, tiles, Hq, Hk, D, short, dt):
    from swiftlm_amd import DFlashKernels as K

    assert (short_splits(1, Hq, Hk, N, D) > 0) == short
    q, k, v = tensors(N + D, 1, Hq, Hk, N, D, dt)
    mask = 0.1 * torch.randn(1, Hq, 16, N, generator=torch.Generator(device="cuda").manual_seed(N), device="cuda")
    for t in tiles:
        mask[..., 32 * t:32 * t + 32] = float("-inf")
    mask[0, 1, 5] = float("-inf")                             # a row without any key
    mask[0, 2, 3] = 0.0                                       # a row that sees the values that are not finite
    mask = mask.to(dt)
    seen = torch.ones(1, Hq, 16, dtype=torch.bool)
    seen[0, 2, 3] = False
    want = O.sdpa_block_causal(host(q), host(k), host(v), 0.1, host(mask).astype(np.float64))
    for t in tiles:
        v[:, :, 32 * t:32 * t + 32] = float("nan")
    out, lse = K.batched_sdpa_2pass(q, k, v, 0.1, mask, return_lse=True)
    same_rows(out[seen], lse[seen], want[0][seen], want[1][seen])
    assert not out[0, 1, 5].any() and torch.isneginf(lse[0, 1, 5])
    assert torch.isnan(out[0, 2, 3]).all()


# ... whoever holds it: a wave of the one workgroup per head or a split of its own, of either form, behind either combine kernel.
# Row r of the block sees keys up to N - 16 + r.
@pytest.mark.parametrize("Hq,Hk,D,N,key", [(4, 2, 128, 33, 32), (4, 2, 256, 33, 32), (3, 1, 128, 300, 299), (3, 1, 256, 300, 31), (16, 2, 256, 1025, 1024),
                                           (16, 2, 256, 4100, 63), (8, 1, 128, 1025, 1024), (8, 1, 128, 8193, 8192), (8, 8, 128, 8193, 703), (64, 8, 256, 4097, 4096),
                                           (520, 8, 128, 97, 96), (520, 8, 128, 300, 290), (264, 8, 256, 97, 96), (264, 8, 256, 300, 290)])
def test_tile_with_only_a_nan_score_is_not_hidden(gpu_lib, Hq, Hk, D, N, key):
    from swiftlm_amd import DFlashKernels as K

    q, k, v = tensors(1, 1, Hq, Hk, N, D)
    k[:, :, key // 32 * 32:key + 1] = float("nan")
    first = max(0, key // 32 * 32 - (N - 16))
    out, lse = K.batched_sdpa_2pass(q, k, v, 0.1, return_lse=True)
    for nan in (torch.isnan(out), torch.isnan(lse)):
        assert nan[:, :, first:].all() and not nan[:, :, :first].any()
    # nothing but NaN
    out, lse = K.batched_sdpa_2pass(q, torch.full_like(k, float("nan")), v, 0.1, return_lse=True)
    assert torch.isnan(out).all() and torch.isnan(lse).all()


# GatedDelta forward with one decay per channel, chunk by chunk: 2 to 6 chunks, whole and ragged last ones, several row tiles; decays of
# zero, of one and below zero among them.  The same steps in calls of 16, which the step kernel takes, are held to the same bounds.
@pytest.mark.parametrize("Dk,Dv,dt", [(64, 16, "bf16"), (128, 48, "bf16"), (128, 16, "f16"), (64, 32, "f16")], ids=lambda v: str(v))
@pytest.mark.parametrize("T", [24, 31, 32, 33, 49, 87])
@pytest.mark.parametrize("masked", [False, True])
def test_channel_gate_chunks(gpu_lib, Dk, Dv, dt, T, masked):
    from swiftlm_amd import DFlashKernels as K

    tdt = {"bf16": torch.bfloat16, "f16": torch.float16}[dt]
    d = O.make_gdn_inputs(Dk + Dv + T, 2, T, 2, 4, Dk, Dv, in_dtype=dt, vec_gate=True)
    d["g"][:, 5::7, :, ::3] = 0.0
    d["g"][:, 3::5, :, 1::4] = 1.0
    d["g"][:, 4::6, :, 2::5] = -0.5
    mask = None
    if masked:
        mask = np.ones((2, T), np.float32)
        mask[0, 2:5] = 0
        mask[0, 15:18] = 0
        mask[1, T - 5:] = 0
    ins = [dev(d[n], tdt) for n in ("q", "k", "v", "g", "beta")]
    dmask = None if mask is None else dev(mask)
    yw, sw, tw = O.gated_delta_ops_with_tape(d["q"], d["k"], d["v"], d["g"], d["beta"], d["state"], mask, dtype=np.float64)

    def run(steps):
        state, parts = dev(d["state"]), []
        for t in range(0, T, steps):
            y, state, tape = K.gated_delta_kernel_with_tape(*[x[:, t:t + steps].contiguous() for x in ins], state,
                                                            None if mask is None else dmask[:, t:t + steps].contiguous())
            parts.append((y, tape))
        return torch.cat([p[0] for p in parts], 1), state, torch.cat([p[1] for p in parts], 1)

    for steps in (T, 16):
        y, s, tape = run(steps)
        np.testing.assert_allclose(host(s), sw, rtol=1e-4, atol=1e-6)
        np.testing.assert_allclose(host(tape), tw, rtol=1e-4, atol=1e-5)
        np.testing.assert_allclose(host(y), yw, rtol=2e-2, atol=2e-2)
        if masked:
            off = mask < 0.5
            assert np.all(host(y)[off] == 0) and np.all(host(tape)[off] == 0)


# The state is as near to 64 bits as the step kernel leaves it, also where decays are fast and the last chunk is a ragged one: the latest
# steps are the largest terms, and each rounding of the sum behind them counts in full.  65,536 values: the ratio of the two errors
# spreads by half a percent.
@pytest.mark.parametrize("T", [29, 36, 42, 64, 78])
@pytest.mark.parametrize("Dk", [64, 128])
def test_channel_gate_state_error(gpu_lib, Dk, T):
    from swiftlm_amd import DFlashKernels as K

    d = O.make_gdn_inputs(Dk + T, 1, T, 4, 8, Dk, 8192 // Dk, in_dtype="bf16", vec_gate=True)
    g = torch.sigmoid(torch.randn(d["g"].shape, generator=torch.Generator().manual_seed(T))).bfloat16()
    d["g"] = g.float().numpy()
    ins = [dev(d[n], torch.bfloat16) for n in ("q", "k", "v", "g", "beta")]
    want = O.gated_delta_ops_with_tape(d["q"], d["k"], d["v"], d["g"], d["beta"], d["state"], dtype=np.float64)[1]

    def error(steps):
        state = dev(d["state"])
        for t in range(0, T, steps):
            state = K.gated_delta_kernel_with_tape(*[x[:, t:t + steps].contiguous() for x in ins], state)[1]
        return np.linalg.norm(host(state).astype(np.float64) - want)

    assert error(T) <= 1.05 * error(16)


# An infinity or NaN of one step stays out of the steps before it (products over all steps of a chunk would spread it), of the other state
# rows and, where the step is masked, out of everything
@pytest.mark.parametrize("what", ["v", "beta", "k_masked", "state"])
def test_channel_gate_not_finite(gpu_lib, what):
    from swiftlm_amd import DFlashKernels as K

    T, t, Dk, Dv = 40, 21, 64, 16
    d = O.make_gdn_inputs(5, 1, T, 1, 2, Dk, Dv, in_dtype="bf16", vec_gate=True)
    mask = np.ones((1, T), np.float32)
    clean = {n: a.copy() for n, a in d.items()}
    if what == "v":
        d["v"][0, t, 1, 3] = np.inf
    elif what == "beta":
        d["beta"][0, t, 1] = np.nan
    elif what == "k_masked":
        d["k"][0, t] = np.inf
        mask[0, t] = 0
    else:
        d["state"][0, 1, 3, 7] = np.nan
    run = lambda x: [host(a) for a in K.gated_delta_kernel_with_tape(*[dev(x[n], torch.bfloat16) for n in ("q", "k", "v", "g", "beta")], dev(x["state"]),
                                                                     dev(mask))]
    y, s, tape = run(d)
    yc, sc, tc = run(clean)
    bad = np.zeros((1, T, 2, Dv), bool)
    rows = slice(None) if what == "beta" else slice(3, 4)
    if what != "k_masked":
        bad[0, 0 if what == "state" else t:, 1, rows] = True
    for got, want in ((y, yc), (tape, tc)):
        np.testing.assert_allclose(got[~bad], want[~bad], rtol=1e-4 if got is tape else 2e-2, atol=1e-5 if got is tape else 2e-2)
        assert not np.isfinite(got[bad]).any()
    hit = bad[0, -1]                                   # [Hv, Dv]
    np.testing.assert_allclose(s[0][~hit], sc[0][~hit], rtol=1e-4, atol=1e-6)
    assert not np.isfinite(s[0][hit]).any()


# A call that one split answers leaves its workspace alone, so that one without a workspace allocates none; both sides of the lines (one split
# for few keys, for many heads and few tiles, and for 4 tiles of keys), counts on the device too
@pytest.mark.parametrize("B,Hq,Hk,D,N,one", [(1, 8, 2, 128, 896, True), (1, 8, 2, 128, 897, False), (1, 32, 8, 128, 1152, True), (1, 32, 8, 128, 1153, False),
                                             (1, 8, 8, 256, 416, True), (1, 8, 8, 256, 417, False), (9, 32, 8, 128, 128, True), (9, 32, 8, 128, 1153, False),
                                             (1, 1, 1, 256, 16, True)], ids=str)
@pytest.mark.parametrize("ragged", [False, True])
def test_attention_scratch(gpu_lib, B, Hq, Hk, D, N, one, ragged):
    from swiftlm_amd import DFlashKernels as K, _lib

    lib = _lib.load()
    need, used = (f(B, Hq, Hk, 16, N, D) for f in (lib.dflash_sdpa_workspace_bytes, lib.dflash_sdpa_scratch_bytes))
    assert used == (0 if one else need) and need > 0
    rng = torch.Generator(device="cuda").manual_seed(N)
    q, k, v = (torch.randn(B, h, n, D, generator=rng, device="cuda").bfloat16() for h, n in ((Hq, 16), (Hk, N), (Hk, N)))
    lens = torch.randint(16, N + 1, (B,), generator=rng, device="cuda", dtype=torch.int32) if ragged else None
    ws = torch.full((need,), 0xA5, dtype=torch.uint8, device="cuda")
    want = K.batched_sdpa_2pass(q, k, v, D ** -0.5, kv_len=lens, return_lse=True, workspace=ws)
    assert bool((ws == 0xA5).all()) == one
    for got, w in zip(K.batched_sdpa_2pass(q, k, v, D ** -0.5, kv_len=lens, return_lse=True), want):
        assert torch.equal(got, w)
    ref = torch.softmax((q.double() @ k.double().repeat_interleave(Hq // Hk, 1).transpose(2, 3).contiguous() * D ** -0.5).masked_fill(
        torch.arange(N, device="cuda") > ((lens if ragged else torch.full((B,), N, device="cuda")).view(B, 1, 1, 1) - 16
                                          + torch.arange(16, device="cuda").view(1, 1, 16, 1)), float("-inf")), -1) @ v.double().repeat_interleave(Hq // Hk, 1)
    np.testing.assert_allclose(host(want[0]), host(ref), rtol=2e-2, atol=2e-2)
