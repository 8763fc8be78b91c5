"""Calls whose q-tiles leave CUs idle run prefill_hilo_kernel with split key ranges and prefill_combine_kernel: against
the oracle at the sizes where the split can go wrong, and bit-identical when repeated.

The outputs' bound is the suite's 2e-3; the projected argmax and the appended cache rows are exact.
"""
import numpy as np
import pytest

import oracle
import workload
from glimpse_language_amd import bonsai_attn as ba

pytestmark = pytest.mark.gpu

# a row short of two q-tiles and one row past; ranges of one, two and three key tiles (unsplit, then split in two);
# q-tiles with different numbers of splits; one kv head with more than 64 splits of one q-tile (the merge's second pass)
# and with more than 64 q-tiles (the block index scan's second pass); a range that ends on a tile's edge
SHAPES = [(63, 0, 8, 2), (65, 0, 8, 2), (66, 30, 8, 2), (96, 0, 16, 4), (100, 300, 8, 2), (65, 5000, 4, 1),
          (2100, 0, 4, 1), (256, 512, 8, 2), (97, 31, 16, 4)]


@pytest.mark.parametrize("T,off,H,KV", SHAPES)
@pytest.mark.parametrize("q16", [False, True])
def test_split_key_ranges(gpu, T, off, H, KV, q16):
    from conftest import context_with
    torch, _, _ = gpu
    print(f"split key ranges T={T} off={off} H={H} KV={KV} fp16 q {q16}", flush=True)
    inp = workload.layer(0x9A00 + T + off, T=T, off=off, H=H, KV=KV)
    if q16:
        inp["q"] = inp["q"].astype(np.float16).astype(np.float32)
    ctx = context_with(BONSAI_ATTN_MID_ROWS=0)  # 63 rows on the q-tiles too
    ws = ba.Workspace(ctx, "cuda")
    dev = {k: torch.from_numpy(np.ascontiguousarray(inp[k])).cuda() for k in ("q", "k_new", "v_new", "gate")}
    q = dev["q"].half() if q16 else dev["q"]
    outs = []
    for _ in range(2):
        kc = torch.from_numpy(inp["kc"].view(np.int16).copy()).cuda()
        vc = torch.from_numpy(inp["vc"].view(np.int16).copy()).cuda()
        out = ba.attention(ctx, ws, q, kc, vc, off, k_new=dev["k_new"], v_new=dev["v_new"], gate=dev["gate"],
                           kind=ba.KIND_PREFILL)
        torch.cuda.synchronize()
        outs.append((out.cpu().numpy(), kc.cpu().numpy().view(np.uint16), vc.cpu().numpy().view(np.uint16)))
    ref, kc_ref, vc_ref = workload.expected(inp)
    assert np.max(np.abs(outs[0][0] - ref)) <= 2e-3
    assert np.array_equal(outs[0][1], kc_ref) and np.array_equal(outs[0][2], vc_ref)
    assert np.array_equal(outs[0][0], outs[1][0]), "repeat call not bit-identical"
    ctx.close()


# merges of at most 8 splits, of 9 to 16, of more than 16 and of more than 64 (the last with one kv head)
@pytest.mark.parametrize("T,off,H,KV", [(256, 512, 8, 2), (70, 512, 16, 4), (96, 1031, 8, 2), (65, 5000, 4, 1)])
@pytest.mark.parametrize("q16", [False, True])
@pytest.mark.parametrize("device_off", [False, True])
def test_split_rotated_in_place_operands(gpu, T, off, H, KV, q16, device_off):
    """Rotated output, with q and the gate read where q_proj leaves them (512 columns a head), the offset from the host or
    from the device below its bound (fewer key tiles than the call's splits are planned for)."""
    from test_gpu_rotate_fused import oracle_rotate, signs_for
    torch, ctx, ws = gpu
    print(f"split rotated T={T} off={off} H={H} KV={KV} fp16 q {q16} device offset {device_off}", flush=True)
    bound = off + 700 if device_off else off
    inp = workload.layer(0x9B00 + T + off, T=T, off=off, H=H, KV=KV, cap=bound + T)
    if q16:
        inp["q"] = inp["q"].astype(np.float16).astype(np.float32)
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    qp = torch.full((T, H, 512), float("nan"), device="cuda")
    qp[:, :, :256], qp[:, :, 256:] = t(inp["q"]), t(inp["gate"])
    qbuf = qp.half() if q16 else qp
    kc, vc = t(inp["kc"].view(np.int16)), t(inp["vc"].view(np.int16))
    signs = signs_for(H)
    st = (H * 512, 512)
    out = ba.attention(ctx, ws, qbuf[:, :, :256], kc, vc, bound, k_new=t(inp["k_new"]), v_new=t(inp["v_new"]),
                       gate=qp[:, :, 256:], kind=ba.KIND_PREFILL, q_strides=st, g_strides=st, signs=t(signs),
                       dyn=torch.tensor([off], dtype=torch.int32, device="cuda") if device_off else None)
    torch.cuda.synchronize()
    ref, kc_ref, vc_ref = workload.expected(inp)
    assert np.max(np.abs(out.cpu().numpy().reshape(T, -1) - oracle_rotate(ref, signs))) <= 2e-3
    assert np.array_equal(kc.cpu().numpy().view(np.uint16), kc_ref)
    assert np.array_equal(vc.cpu().numpy().view(np.uint16), vc_ref)
