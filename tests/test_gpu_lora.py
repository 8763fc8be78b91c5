"""The LoRA down projection rows (u = A x, kernels/rot.glsl:19-40 LORA_ROW) of bn_gate_rotate, bn_norm_rotate and the
attention calls, on the GPU.

bn_gate_rotate and bn_norm_rotate compute them in extra blocks of their launch: u is checked against the oracle's
LORA_ROW restatement (x = attn * sigmoid(gate), or the normed row), within 1e-6 of sum |A x| (fp32 sums in another
order), and the rotated output is unchanged by the extra blocks. After an attention call the rows come from the
call's own output: u is checked against A times that output's gated rows recovered on the host in float64 (the
inverse rotation s * H xr / sqrt(512)), within 1e-5 of sum |A x|, and against the oracle's attention within
2e-3 * sum |A| (the attention bar carried through A).
"""
import numpy as np
import pytest
import scipy.linalg

import oracle
import workload
from glimpse_language_amd import bonsai_attn as ba
from test_gpu_prep_rotate import inv_freq, prep_inputs, oracle_prep, to_dev as dev

pytestmark = pytest.mark.gpu
D = 256


def lora_a(seed, R, K):
    return oracle.f32_to_f16(oracle.normal(seed, 20, (R, K)) * np.float32(0.05))


def bound(A, x, rel):
    return rel * (np.abs(x.astype(np.float64)) @ np.abs(oracle.f16_to_f32(A).astype(np.float64)).T) + 1e-7


@pytest.mark.parametrize("T,H,R", [(1, 16, 48), (5, 8, 7), (100, 16, 16), (3, 32, 33)])
def test_gate_rotate_lora_rows(gpu, T, H, R):
    torch, ctx, _ = gpu
    W = H * D
    attn = oracle.normal(0x1A00 + T, 0, (T, W))
    qp = oracle.normal(0x1A00 + T, 1, (T, H, 512))
    s = np.where(oracle.normal(0x1A00 + T, 2, (W,)) > 0, 1.0, -1.0).astype(np.float32)
    A = lora_a(0x1A00 + T, R, W)
    qpd = dev(torch, qp)
    u = torch.full((T, R), float("nan"), device="cuda")
    xr = ba.gate_rotate(ctx, dev(torch, attn), dev(torch, s), gate=qpd[:, :, D:], lora=(dev(torch, A), u))
    plain = ba.gate_rotate(ctx, dev(torch, attn), dev(torch, s), gate=qpd[:, :, D:])
    torch.cuda.synchronize()
    ref = oracle.lora_gate(A, attn, qp)
    x = attn.astype(np.float64) / (1.0 + np.exp(-qp[:, :, D:].reshape(T, W).astype(np.float64)))
    got = u.cpu().numpy()
    assert np.all(np.abs(got - ref) <= bound(A, x, 1e-6)), np.max(np.abs(got - ref))
    assert np.array_equal(xr.cpu().numpy(), plain.cpu().numpy())


@pytest.mark.parametrize("T,Dm,R", [(1, 2560, 48), (7, 2048, 24), (100, 2560, 16), (2, 8192, 5)])
def test_norm_rotate_lora_rows(gpu, T, Dm, R):
    torch, ctx, _ = gpu
    h = oracle.normal(0x1B00 + T, 0, (T, Dm)) * np.float32(2.0)
    w = (1.0 + 0.1 * oracle.normal(0x1B00 + T, 1, (Dm,))).astype(np.float32)
    s = np.where(oracle.normal(0x1B00 + T, 2, (Dm,)) > 0, 1.0, -1.0).astype(np.float32)
    A = lora_a(0x1B00 + T, R, Dm)
    u = torch.full((T, R), float("nan"), device="cuda")
    xn = torch.empty((T, Dm), device="cuda")
    xr = ba.norm_rotate(ctx, dev(torch, h), dev(torch, w), dev(torch, s), xn=xn, lora=(dev(torch, A), u))
    plain = ba.norm_rotate(ctx, dev(torch, h), dev(torch, w), dev(torch, s))
    torch.cuda.synchronize()
    _, ref_xn = oracle.norm_rotate(h, w, s, want_xn=True)
    ref = oracle.lora(A, ref_xn)
    got = u.cpu().numpy()
    assert np.all(np.abs(got - ref) <= bound(A, ref_xn, 1e-6)), np.max(np.abs(got - ref))
    # the extra blocks norm the rows as the main blocks do: u equals the LoRA rows of the written xn within rounding
    xg = xn.cpu().numpy()
    assert np.all(np.abs(got - oracle.lora(A, xg)) <= bound(A, xg, 1e-6))
    assert np.array_equal(xr.cpu().numpy(), plain.cpu().numpy())


def unrotate(xr, signs):
    """float64 inverse of the rotation: per 512-block, s * H xr / sqrt(512)."""
    T, W = xr.shape
    Hm = scipy.linalg.hadamard(512).astype(np.float64)
    y = xr.astype(np.float64).reshape(T, W // 512, 512) @ Hm / np.sqrt(512.0)
    return y.reshape(T, W) * signs.astype(np.float64)


# (T, off, H, KV, kind, rotated): decode, verify rows on the MFMA kernel, a prefill, each with and without rotation
@pytest.mark.parametrize("T,off,H,KV,kind,rot", [
    (1, 3000, 16, 4, ba.KIND_DECODE, True), (1, 500, 8, 2, ba.KIND_DECODE, False),
    (8, 2048, 8, 2, ba.KIND_VERIFY, True), (100, 300, 16, 4, ba.KIND_PREFILL, True),
    (40, 0, 8, 2, ba.KIND_PREFILL, False),
])
def test_attention_lora_rows(gpu, T, off, H, KV, kind, rot):
    torch, ctx, ws = gpu
    R, W = 12, H * D
    inp = workload.layer(0x1C00 + T + off, T=T, off=off, H=H, KV=KV)
    s = np.where(oracle.normal(0x1C00 + T, 3, (W,)) > 0, 1.0, -1.0).astype(np.float32) if rot else None
    A = lora_a(0x1C00 + T, R, W)
    t = lambda x: None if x is None else torch.from_numpy(np.ascontiguousarray(x)).cuda()
    u = torch.full((T, R), float("nan"), device="cuda")
    out = ba.attention(ctx, ws, t(inp["q"]), t(inp["kc"].view(np.int16)), t(inp["vc"].view(np.int16)), off,
                       k_new=t(inp["k_new"]), v_new=t(inp["v_new"]), gate=t(inp["gate"]), kind=kind, signs=t(s),
                       lora=(t(A.view(np.int16)), u))
    torch.cuda.synchronize()
    o = out.cpu().numpy().reshape(T, W)
    g = unrotate(o, s) if rot else o.astype(np.float64)
    got = u.cpu().numpy()
    ref_gpu = g @ oracle.f16_to_f32(A).astype(np.float64).T
    assert np.all(np.abs(got - ref_gpu) <= bound(A, g, 1e-5)), np.max(np.abs(got - ref_gpu))
    ref_attn, _, _ = workload.expected(inp)
    ref = oracle.lora(A, ref_attn.reshape(T, W))
    assert np.all(np.abs(got - ref) <= 2e-3 * np.abs(oracle.f16_to_f32(A)).sum(axis=1)[None, :])


# (T, off, H, KV): a decode step, 8 verify rows (prep_kernel, then verify_kernel), a prefill (prep_kernel writes the
# q scratch, prefill_hilo_kernel with split keys, the rotation in the merge)
@pytest.mark.parametrize("T,off,H,KV", [(1, 2047, 16, 4), (8, 1000, 8, 2), (100, 300, 8, 2)])
def test_layer_lora_rows(gpu, T, off, H, KV):
    """bn_attn_layer (the whole arm, rotated) with the LoRA rows: u from the call's own output, and vs the oracle."""
    torch, ctx, ws = gpu
    R = 8
    seed = 0x1D00 + T
    inp = prep_inputs(seed, T, off, H, KV)
    W = H * D
    s = np.where(oracle.normal(seed, 9, (W,)) > 0, 1.0, -1.0).astype(np.float32)
    A = lora_a(seed, R, W)
    print(f"layer lora rows: T={T} off={off} H={H} KV={KV}", flush=True)
    d = {k: dev(torch, inp[k]) for k in ("qp", "kp", "vp", "qn", "kn", "pos", "inv", "kc", "vc")}
    u = torch.full((T, R), float("nan"), device="cuda")
    out = ba.attention_layer(ctx, ws, d["qp"], d["kp"], d["vp"], d["qn"], d["kn"], d["pos"], d["inv"], d["kc"],
                             d["vc"], off, gate=d["qp"][:, :, D:], signs=dev(torch, s), lora=(dev(torch, A), u))
    torch.cuda.synchronize()
    g = unrotate(out.cpu().numpy().reshape(T, W), s)
    ref_gpu = g @ oracle.f16_to_f32(A).astype(np.float64).T
    got = u.cpu().numpy()
    assert np.all(np.abs(got - ref_gpu) <= bound(A, g, 1e-5))
    q_ref, kc_ref, vc_ref = oracle_prep(inp)
    attn = oracle.attend(q_ref, kc_ref, vc_ref, off, inp["qp"][:, :, D:]).reshape(T, W)
    assert np.all(np.abs(got - oracle.lora(A, attn)) <= 2e-3 * np.abs(oracle.f16_to_f32(A)).sum(axis=1)[None, :])


def test_lora_argument_checks(gpu):
    torch, ctx, _ = gpu
    T, H = 2, 8
    attn = torch.zeros((T, H * D), device="cuda")
    s = torch.ones(H * D, device="cuda")
    A = torch.zeros((4, H * D), dtype=torch.int16, device="cuda")
    u = torch.zeros((T, 4), device="cuda")
    a = ba.rotate_args(attn, s, attn, lora=(A, u))  # in place with LoRA rows: rejected
    assert ba.check(a) == ba.BN_EINVAL
    a = ba.rotate_args(attn, s, torch.zeros_like(attn), lora=(A, u))
    assert ba.check(a) == ba.BN_OK
    a.lora_us = 2                                     # rows of u shorter than lora_r
    assert ba.check(a) == ba.BN_EINVAL
