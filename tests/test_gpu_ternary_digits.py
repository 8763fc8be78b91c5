"""bn_ternary_matmul with more than 32 tokens (bn_ternary_mx.h) against float64: x as five base-32 digits per block of 32
columns of a token, with a second set where columns of a block lie far below its largest.

Bound per output, from the arithmetic: a block's digits end within 2^-24 of its largest value (where 12 or more columns
lie 2^6 below that, it has a second set: 2^-24 of the remainder's, so 2^-44), and each group's sum takes at most 20 additions of MFMA
results and one fma, each rounding the running sum by at most 2^-23 of sum |x w| (2^-24 for one rounding, doubled for an
accumulation inside the MFMA); the groups' sums add one more each.
"""
import numpy as np
import pytest

import oracle
import workload
from glimpse_language_amd import bonsai_attn as ba

pytestmark = pytest.mark.gpu


def dev(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def call(torch, ctx, mats, x, work):
    xd = dev(torch, x)
    ys = [torch.full((x.shape[0], w.shape[0]), float("nan"), device="cuda") for w, _, _ in mats]
    ws = ba.ternary_workspace(xd) if work else None
    if work:
        ws.fill_(0xA5)
    ba.ternary_matmul(ctx, xd, [(dev(torch, w.view(np.int32)), dev(torch, s.view(np.int16)), y)
                                for (w, s, _), y in zip(mats, ys)], work=ws)
    torch.cuda.synchronize()
    return [y.cpu().numpy() for y in ys]


def exact(w, s, codes, x):
    full = (codes.astype(np.float64) - 1) * np.repeat(oracle.f16_to_f32(s).astype(np.float64), 128, axis=1)
    x = x.astype(np.float64)
    blocks = np.abs(x).reshape(x.shape[0], -1, 32)
    mx = blocks.max(-1)
    cut = np.where((blocks <= mx[..., None] / 64).sum(-1) >= 12, 2.0 ** -44, 2.0 ** -24) * mx
    aw = np.abs(full)
    split = cut @ aw.reshape(aw.shape[0], -1, 32).sum(-1).T
    groups = x.shape[1] // 128
    return x @ full.T, split + (21 + groups) * 2.0 ** -23 * (np.abs(x) @ aw.T)


# tokens at the edges of the 32- and 64-token tiles; one group (the second wave group has it alone), three (odd, scales
# one at a time), rows that leave 128- and 256-row blocks partly empty; 32 x 256 blocks; 64 x 256 blocks
SHAPES = [(33, 128, (64,)), (64, 384, (192,)), (65, 512, (320, 64)), (97, 2048, (128,)), (500, 256, (4096, 512, 512)),
          (1025, 256, (4096, 512, 512))]


@pytest.mark.parametrize("T,K,os", SHAPES)
def test_digits_against_float64(gpu, T, K, os):
    torch, ctx, _ = gpu
    print(f"ternary digits T={T} K={K} os={os}", flush=True)
    mats = [workload.ternary_weights(0x7A00 + T + i, o, K, True) for i, o in enumerate(os)]
    x = oracle.normal(0x7A00 + T, 1, (T, K)).copy()
    # blocks that need a second set (in the first, a middle and the last token), a block of one value and zeros, tiny
    # values, values whose digits end early
    x[0, 5], x[T // 2, K - 1], x[T - 1, 40] = 3.0e4, -1.0e7, 700.0
    x[1, :32] = 0.0
    x[1, 3] = 1.1
    x[2] *= 2.0 ** -60
    x[3] = np.round(x[3] * 4)
    got = call(torch, ctx, mats, x, True)
    for g, (w, s, codes) in zip(got, mats):
        ref, tol = exact(w, s, codes, x)
        bad = np.argwhere(~(np.abs(g - ref) <= tol))
        assert bad.size == 0, f"{len(bad)} outputs off, first {bad[:3].tolist()}"
    assert all(np.array_equal(a, b) for a, b in zip(got, call(torch, ctx, mats, x, False))), "without a workspace"


def test_digits_nonfinite_token(gpu):
    """An infinity or a NaN makes its own token's outputs NaN and leaves the others as they are."""
    torch, ctx, _ = gpu
    T, K, os = 70, 384, (128,)
    mats = [workload.ternary_weights(0x7B00, os[0], K, False)]
    x = oracle.normal(0x7B00, 1, (T, K)).copy()
    clean = call(torch, ctx, mats, x, True)[0]
    x[4, 200], x[66, 0] = np.inf, np.nan
    for work in (True, False):
        got = call(torch, ctx, mats, x, work)[0]
        assert np.isnan(got[[4, 66]]).all()
        rest = np.setdiff1d(np.arange(T), [4, 66])
        assert np.array_equal(got[rest], clean[rest])


@pytest.mark.parametrize("large,mag", [(5, 1e3), (6, 1e4), (8, 30.0), (8, 2e4), (16, 300.0), (20, 60.0), (24, 100.0),
                                       (24, 1e3), (24, 1e5)])
def test_small_columns_beside_large_ones(gpu, large, mag):
    """Some columns of every 32 (the same for all tokens, as channels of another scale are) hold values mag times the
    others', under weights 0: what is left are the small columns' products, to workload.ternary_tolerance (2e-5 of their
    norm) as for any other call. Then with the large values in one token of 16 only."""
    torch, ctx, _ = gpu
    T, K, O = 70, 768, 256
    w, s, codes = workload.ternary_weights(0x7C00 + large, O, K, True)
    rank = np.argsort(np.argsort(oracle.normal(0x7C00 + large, 2, (K // 32, 32)), axis=1), axis=1).reshape(-1)
    big = rank < large
    codes[:, big] = 1
    w = workload.pack_codes(codes)
    base = oracle.normal(0x7C00 + large, 1, (T, K)).copy()
    for tokens in (np.arange(T), np.arange(3, T, 16)):
        print(f"ternary digits, {large} of 32 columns x {mag} in {len(tokens)} tokens", flush=True)
        x = base.copy()
        x[np.ix_(tokens, big)] *= np.float32(mag)
        full = (codes.astype(np.float64) - 1) * np.repeat(oracle.f16_to_f32(s).astype(np.float64), 128, axis=1)
        ref, tol = x.astype(np.float64) @ full.T, workload.ternary_tolerance(x, codes, s)
        for work in (True, False):
            got = call(torch, ctx, [(w, s, codes)], x, work)[0]
            worst = float(np.max(np.abs(got - ref) / tol))
            assert worst <= 1, f"workspace {work}: {worst:.2f} of the bound"


# without a workspace: 32 x 512 blocks (an odd number of groups, rows of three matrices), 64 x 512 blocks, full rounds of
# those and 32 x 512 blocks for the last 100 tokens, and for the last one
@pytest.mark.parametrize("T,K", [(700, 384), (1025, 128), (1700, 256), (1601, 128)])
def test_in_place_blocks(gpu, T, K):
    """Calls that add into strided outputs, with LoRA rows and a strided x: the same bits with and without a workspace,
    and within workload.ternary_tolerance of float64 (and of 1e-6 of the LoRA part, 16 fp32 products)."""
    torch, ctx, _ = gpu
    os, r, pad = (4096, 512, 512), 16, 8
    print(f"ternary in place T={T} K={K}", flush=True)
    mats = [workload.ternary_weights(0x7D00 + i, o, K, True) for i, o in enumerate(os)]
    x = oracle.normal(0x7D00 + T, 1, (T, K + pad)).copy()
    y0 = [oracle.normal(0x7D10 + i, 2, (T, o + 4)) for i, o in enumerate(os)]
    lu = oracle.normal(0x7D20, 3, (T, 3 * r + 5))
    lb = [oracle.f32_to_f16(oracle.normal(0x7D30 + i, 4, (o, r))) for i, o in enumerate(os)]
    xd, lud = dev(torch, x)[:, :K], dev(torch, lu)
    packed = [(dev(torch, w.view(np.int32)), dev(torch, s.view(np.int16))) for w, s, _ in mats]
    lbd = [dev(torch, b.view(np.int16)) for b in lb]
    got = []
    for work in (True, False):
        ys = [dev(torch, y) for y in y0]
        ba.ternary_matmul(ctx, xd, [(w, s, y[:, :o], b) for (w, s), y, o, b in zip(packed, ys, os, lbd)], add=True,
                          lora_u=lud, lora_r=r, work=ba.ternary_workspace(xd) if work else None)
        torch.cuda.synchronize()
        got.append([y.cpu().numpy() for y in ys])
    for i, ((w, s, codes), o) in enumerate(zip(mats, os)):
        a, b = got[0][i], got[1][i]
        assert np.array_equal(a, b), f"matrix {i}"
        assert np.array_equal(a[:, o:], y0[i][:, o:]), "columns beside the matrix"
        full = (codes.astype(np.float64) - 1) * np.repeat(oracle.f16_to_f32(s).astype(np.float64), 128, axis=1)
        u, B = lu[:, i * r:(i + 1) * r].astype(np.float64), oracle.f16_to_f32(lb[i]).astype(np.float64)
        ref = x[:, :K].astype(np.float64) @ full.T + u @ B.T + y0[i][:, :o]
        tol = workload.ternary_tolerance(x[:, :K], codes, s) + 1e-6 * (np.abs(u) @ np.abs(B).T + np.abs(y0[i][:, :o]))
        assert (np.abs(a[:, :o] - ref) <= tol).all(), f"matrix {i}"
