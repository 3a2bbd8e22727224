"""a9/a10 expert product + combine vs the oracle.  Align plan bit-exact;
outputs within rel-L2 1e-2 (bf16 weights) and 3e-2 (fp8 e4m3fn weights,
128x128 block scales), the tolerances the path is specified to."""

import ctypes

import numpy as np
import pytest
import torch

from oracle import moe as om

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")
BF16_TOL = 1e-2
FP8_TOL = 3e-2


def _routing(T, E, k, rng):
    return np.stack([rng.choice(E, size=k, replace=False) for _ in range(T)]).astype(np.int32)


def _emap(E, S, rng, resident_frac=1.0):
    """global -> slot map with S resident experts (some selected ids may miss)."""
    emap = np.full(E, -1, np.int32)
    res = rng.choice(E, size=S, replace=False)
    for s, g in enumerate(res):
        if rng.random() < resident_frac:
            emap[g] = s
    return emap


def _bf16(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).to(torch.bfloat16)


@pytest.mark.parametrize("T,k,E,S,seed", [(1, 6, 64, 48, 0), (8, 6, 64, 48, 1), (12, 8, 128, 96, 2),
                                          (40, 4, 16, 8, 3), (300, 8, 64, 64, 4), (0, 8, 64, 8, 5)])
def test_align_plan_bit_exact(T, k, E, S, seed):
    from sluice_amd import _lib

    lib = _lib.load()
    rng = np.random.default_rng(seed)
    ids = _routing(T, E, k, rng) if T else np.zeros((0, k), np.int32)
    emap = _emap(E, S, rng, resident_frac=0.8)
    ids[0:1, 0:1] = E + 3 if T else 0  # an out-of-range id is simply invalid
    n = _lib.load().sluice_moe_plan_ints(max(T, 1), k)
    plan = torch.full((n,), -7, dtype=torch.int32, device=DEV)
    ids_d = torch.from_numpy(ids).to(DEV)
    emap_d = torch.from_numpy(emap).to(DEV)
    rc = lib.sluice_moe_align(ids_d.data_ptr(), T, k, emap_d.data_ptr(), E, S, plan.data_ptr(),
                              torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "align")
    torch.cuda.synchronize()
    p = plan.cpu().numpy()
    print(f"align T={T} k={k} E={E} S={S}", flush=True)
    blocks, valid = om.align_blocks(ids, emap, S, 16)
    assert p[0] == len(blocks)
    assert p[2] == len(blocks)  # no slot of this map streams: every block is resident
    if T == 0:
        return
    P = T * k
    for b, (slot, pairs) in enumerate(blocks):
        rec = p[4 + 18 * b: 4 + 18 * (b + 1)]
        assert rec[0] == slot and rec[1] == len(pairs)
        assert rec[2:2 + len(pairs)].tolist() == pairs
    assert p[4 + 18 * P: 4 + 19 * P].tolist() == valid


def _moe_case(T, H, I, E, S, k, seed, resident_frac=0.85, use_map=True, scale=1.0, shared=False):
    from sluice_amd import ops

    rng = np.random.default_rng(seed)
    x = _bf16(rng.standard_normal((T, H)))
    w13 = _bf16(rng.standard_normal((S, 2 * I, H)) * 0.02)
    w2 = _bf16(rng.standard_normal((S, H, I)) * 0.02)
    ids = _routing(T, E if use_map else S, k, rng)
    tw = rng.random((T, k)).astype(np.float32)
    emap = _emap(E, S, rng, resident_frac) if use_map else None
    sh = _bf16(rng.standard_normal((T, H))) if shared else None
    out = ops.fused_experts(
        x.to(DEV), w13.to(DEV), w2.to(DEV), torch.from_numpy(tw).to(DEV),
        torch.from_numpy(ids).to(DEV), activation="silu",
        global_num_experts=E, expert_map=None if emap is None else torch.from_numpy(emap).to(DEV),
        routed_scaling_factor=scale, shared_output=None if sh is None else sh.to(DEV))
    torch.cuda.synchronize()
    ref = om.fused_experts(x.float().numpy(), w13.float().numpy(), w2.float().numpy(), tw, ids,
                           expert_map=emap, scale=scale,
                           shared=None if sh is None else sh.float().numpy())
    return out.float().cpu().numpy(), ref


@pytest.mark.parametrize("T,H,I,E,S,k", [
    (1, 2048, 1408, 64, 8, 6),      # V2-Lite expert shape, c=1
    (8, 2048, 1408, 64, 12, 6),     # V2-Lite c=8
    (1, 2048, 768, 128, 8, 8),      # Qwen3 c=1
    (8, 2048, 768, 128, 16, 8),     # Qwen3 c=8
    (12, 2048, 768, 128, 16, 8),    # Qwen3 c=12
    (8, 4096, 14336, 8, 2, 2),      # Mixtral-8x7B expert shape (top-2, long K in gemm2)
    (8, 5120, 1536, 160, 8, 6),     # DeepSeek-V2 (236B) expert shape
    (8, 2048, 1024, 64, 16, 8),     # OLMoE-1B-7B expert shape
    (8, 2048, 1408, 60, 16, 4),     # Qwen1.5-MoE-A2.7B expert shape (60 experts)
    (33, 256, 192, 16, 16, 4),      # > 16 pairs per slot: several blocks per expert
    (5, 64, 128, 8, 8, 2),          # K shorter than the waves: some waves stream nothing
    (120, 1088, 448, 40, 40, 5),    # the tiled kernels, 64-pair tiles
    (900, 1088, 448, 40, 40, 5),    # 128-pair tiles, over 4096 pairs
])
def test_fused_experts_bf16(T, H, I, E, S, k):
    print(f"fused bf16 T={T} H={H} I={I} E={E} S={S} k={k}", flush=True)
    got, ref = _moe_case(T, H, I, E, S, k, seed=T * 7 + I)
    err = om.rel_l2(got, ref)
    print(f"  rel_l2={err:.2e}", flush=True)
    assert err <= BF16_TOL


def test_fused_experts_bf16_large_batch():
    """A prefill-sized call (40 tokens, 320 pairs)."""
    got, ref = _moe_case(40, 256, 64, 32, 16, 8, seed=21)
    assert om.rel_l2(got, ref) <= BF16_TOL


def test_fused_experts_deterministic():
    """Identical calls give identical bits (every pair's sum is reduced in a
    fixed order), and the result matches the oracle."""
    from sluice_amd import ops

    rng = np.random.default_rng(5)
    T, H, I, E, S, k = 8, 2048, 768, 128, 32, 8
    x = _bf16(rng.standard_normal((T, H))).to(DEV)
    w13 = _bf16(rng.standard_normal((S, 2 * I, H)) * 0.02).to(DEV)
    w2 = _bf16(rng.standard_normal((S, H, I)) * 0.02).to(DEV)
    ids = torch.from_numpy(_routing(T, E, k, rng)).to(DEV)
    emap = torch.from_numpy(_emap(E, S, rng, 0.9)).to(DEV)
    tw = torch.rand((T, k), device=DEV)
    outs = [ops.fused_experts(x, w13, w2, tw, ids, global_num_experts=E, expert_map=emap)
            for _ in range(3)]
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[1], outs[2])
    ref = om.fused_experts(x.float().cpu().numpy(), w13.float().cpu().numpy(),
                           w2.float().cpu().numpy(), tw.cpu().numpy(), ids.cpu().numpy(),
                           expert_map=emap.cpu().numpy())
    assert om.rel_l2(outs[0].float().cpu().numpy(), ref) <= BF16_TOL


def _staged(lib, x, w13, w2, tw, ids, emap, T, H, I, E, S, k, scale, sh, st, fp8=None):
    """align -> gemm1 -> gemm2 -> combine, one stage entry point at a time."""
    P = T * k
    plan = torch.empty(lib.sluice_moe_plan_ints(T, k), dtype=torch.int32, device=DEV)
    act = torch.empty((P, I), dtype=torch.bfloat16, device=DEV)
    part = torch.empty((P, H), dtype=torch.float32, device=DEV)
    out = torch.empty((T, H), dtype=torch.bfloat16, device=DEV)
    assert lib.sluice_moe_align(ids.data_ptr(), T, k, emap.data_ptr(), E, S, plan.data_ptr(),
                                st) == 0
    if fp8 is None:
        assert lib.sluice_moe_gemm1_bf16(x.data_ptr(), w13.data_ptr(), plan.data_ptr(), T, H, I,
                                         k, act.data_ptr(), st) == 0
        assert lib.sluice_moe_gemm2_bf16(act.data_ptr(), w2.data_ptr(), plan.data_ptr(),
                                         tw.data_ptr(), T, H, I, k, part.data_ptr(), st) == 0
    else:
        s13, s2 = fp8
        assert lib.sluice_moe_gemm1_fp8(x.data_ptr(), w13.data_ptr(), s13.data_ptr(),
                                        plan.data_ptr(), T, H, I, k, act.data_ptr(), st) == 0
        assert lib.sluice_moe_gemm2_fp8(act.data_ptr(), w2.data_ptr(), s2.data_ptr(),
                                        plan.data_ptr(), tw.data_ptr(), T, H, I, k,
                                        part.data_ptr(), st) == 0
    assert lib.sluice_moe_combine(part.data_ptr(), plan.data_ptr(), T, k, H, scale,
                                  None if sh is None else sh.data_ptr(), out.data_ptr(), st) == 0
    return out


@pytest.mark.parametrize("T,H,I,E,S,k,frac,shared,fp8", [
    (8, 2048, 1408, 64, 48, 6, 0.85, True, False),   # V2-Lite shape, shared expert added
    (12, 2048, 768, 128, 96, 8, 0.85, False, False),  # Qwen3 shape
    (33, 256, 192, 16, 16, 4, 0.85, False, False),   # several blocks per slot
    (4, 256, 64, 32, 4, 2, 0.0, True, False),        # nothing resident: out = shared
    (8, 7168, 2048, 256, 12, 8, 0.85, True, True),   # V3 shape, fp8 + block scales
])
def test_fused_experts_matches_its_stages(T, H, I, E, S, k, frac, shared, fp8):
    """fused_experts gives the bits of its stages run one entry point at a
    time (align, gemm1, gemm2, combine), on every call."""
    from sluice_amd import _lib, ops

    lib = _lib.load()
    rng = np.random.default_rng(T * 13 + I)
    x = _bf16(rng.standard_normal((T, H))).to(DEV)
    kw, scales = {}, None
    if fp8:
        def codes(shape):  # e4m3fn codes without the two NaN encodings
            q = rng.integers(0, 256, size=shape, dtype=np.uint8)
            q[(q & 0x7F) == 0x7F] = 0x38
            return torch.from_numpy(q).to(DEV)

        w13, w2 = codes((S, 2 * I, H)), codes((S, H, I))
        scales = (torch.rand((S, 2 * I // 128, H // 128), device=DEV) * 0.02 + 0.01,
                  torch.rand((S, H // 128, I // 128), device=DEV) * 0.02 + 0.01)
        kw = dict(w1_scale=scales[0], w2_scale=scales[1], block_shape=[128, 128])
    else:
        w13 = _bf16(rng.standard_normal((S, 2 * I, H)) * 0.02).to(DEV)
        w2 = _bf16(rng.standard_normal((S, H, I)) * 0.02).to(DEV)
    ids = torch.from_numpy(_routing(T, E, k, rng)).to(DEV)
    emap = torch.from_numpy(_emap(E, S, rng, frac)).to(DEV)
    tw = torch.rand((T, k), device=DEV)
    sh = _bf16(rng.standard_normal((T, H))).to(DEV) if shared else None
    st = torch.cuda.current_stream().cuda_stream
    ref = _staged(lib, x, w13, w2, tw, ids, emap, T, H, I, E, S, k, 1.5, sh, st, fp8=scales)
    for rep in range(3):
        got = ops.fused_experts(x, w13, w2, tw, ids, global_num_experts=E, expert_map=emap,
                                routed_scaling_factor=1.5, shared_output=sh, **kw)
        torch.cuda.synchronize()
        assert torch.equal(got, ref), f"call {rep}"
    if frac == 0.0:
        assert torch.equal(ref, sh)


@pytest.mark.parametrize("T,H,I,Is,E,S,k,frac,fp8", [
    (8, 2048, 1408, 2816, 64, 48, 6, 0.85, False),   # V2-Lite: 2 shared experts
    (1, 2048, 1408, 2816, 64, 48, 6, 0.85, False),
    (20, 256, 64, 192, 16, 8, 4, 0.85, False),       # > 16 tokens: two shared blocks each
    (4, 256, 64, 128, 32, 4, 2, 0.0, False),         # nothing routed resident: shared only
    (8, 7168, 2048, 2048, 256, 12, 8, 0.85, True),   # DeepSeek-V3: 1 fp8 shared expert
])
def test_fused_experts_with_shared_experts(T, H, I, Is, E, S, k, frac, fp8):
    """Shared experts inside the grouped product (shared_w1/shared_w2, Is/I
    groups of I channels, added unscaled) against the oracle's routed sum
    times the routed scale plus the SwiGLU shared MLP; repeated calls give the
    same bits."""
    from sluice_amd import ops

    rng = np.random.default_rng(T * 31 + Is)
    x = _bf16(rng.standard_normal((T, H)))
    ids = _routing(T, E, k, rng)
    tw = rng.random((T, k)).astype(np.float32)
    emap = _emap(E, S, rng, frac)
    if fp8:
        def codes(shape):
            q = rng.integers(0, 256, size=shape, dtype=np.uint8)
            q[(q & 0x7F) == 0x7F] = 0x38
            return q

        def scales(shape):
            return (rng.random(shape) * 0.02 + 0.01).astype(np.float32)

        q13, q2 = codes((S, 2 * I, H)), codes((S, H, I))
        s13, s2 = scales((S, 2 * I // 128, H // 128)), scales((S, H // 128, I // 128))
        qgu, qd = codes((2 * Is, H)), codes((H, Is))
        sgu, sd = scales((2 * Is // 128, H // 128)), scales((H // 128, Is // 128))
        w13, w2 = om.dequant_block(q13, s13), om.dequant_block(q2, s2)
        gu, d = om.dequant_block(qgu, sgu), om.dequant_block(qd, sd)
        args = [torch.from_numpy(a).to(DEV) for a in (q13, q2, qgu, qd)]
        kw = dict(w1_scale=torch.from_numpy(s13).to(DEV), w2_scale=torch.from_numpy(s2).to(DEV),
                  block_shape=[128, 128], shared_w1=args[2], shared_w2=args[3],
                  shared_w1_scale=torch.from_numpy(sgu).to(DEV),
                  shared_w2_scale=torch.from_numpy(sd).to(DEV))
        tol = FP8_TOL
    else:
        w13 = _bf16(rng.standard_normal((S, 2 * I, H)) * 0.02)
        w2 = _bf16(rng.standard_normal((S, H, I)) * 0.02)
        gu = _bf16(rng.standard_normal((2 * Is, H)) * 0.02)
        d = _bf16(rng.standard_normal((H, Is)) * 0.02)
        args = [w13.to(DEV), w2.to(DEV)]
        kw = dict(shared_w1=gu.to(DEV), shared_w2=d.to(DEV))
        w13, w2, gu, d = (a.float().numpy() for a in (w13, w2, gu, d))
        tol = BF16_TOL
    outs = [ops.fused_experts(x.to(DEV), args[0], args[1], torch.from_numpy(tw).to(DEV),
                              torch.from_numpy(ids).to(DEV), global_num_experts=E,
                              expert_map=torch.from_numpy(emap).to(DEV),
                              routed_scaling_factor=2.5, **kw) for _ in range(2)]
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1])
    xf = x.float().numpy()
    ref = om.fused_experts(xf, w13, w2, tw, ids, expert_map=emap, scale=2.5,
                           shared=om.shared_mlp(xf, gu, d))
    err = om.rel_l2(outs[0].float().cpu().numpy(), ref)
    print(f"shared fold T={T} I={I} Is={Is} fp8={fp8}: rel_l2={err:.2e}", flush=True)
    assert err <= tol


def test_fused_experts_rejects_shared_not_a_multiple_of_I():
    from sluice_amd import ops

    x = torch.zeros((2, 256), dtype=torch.bfloat16, device=DEV)
    w13 = torch.zeros((4, 128, 256), dtype=torch.bfloat16, device=DEV)
    w2 = torch.zeros((4, 256, 64), dtype=torch.bfloat16, device=DEV)
    with pytest.raises(ValueError):
        ops.fused_experts(x, w13, w2, torch.ones((2, 2), device=DEV),
                          torch.zeros((2, 2), dtype=torch.int32, device=DEV),
                          shared_w1=torch.zeros((192, 256), dtype=torch.bfloat16, device=DEV),
                          shared_w2=torch.zeros((256, 96), dtype=torch.bfloat16, device=DEV))


def test_fused_experts_bf16_identity_map_scale_shared():
    got, ref = _moe_case(8, 512, 128, 8, 8, 2, seed=9, use_map=False, scale=2.5, shared=True)
    assert om.rel_l2(got, ref) <= BF16_TOL


def test_fused_experts_all_unmapped_is_zero():
    got, ref = _moe_case(4, 256, 64, 32, 4, 2, seed=11, resident_frac=0.0)
    assert np.all(got == 0) and np.all(ref == 0)


def test_fused_experts_empty():
    from sluice_amd import ops

    x = torch.zeros((0, 256), dtype=torch.bfloat16, device=DEV)
    w13 = torch.zeros((2, 128, 256), dtype=torch.bfloat16, device=DEV)
    w2 = torch.zeros((2, 256, 64), dtype=torch.bfloat16, device=DEV)
    out = ops.fused_experts(x, w13, w2, torch.zeros((0, 2), device=DEV),
                            torch.zeros((0, 2), dtype=torch.int32, device=DEV))
    assert out.shape == (0, 256)


def _fp8_case(T, H, I, E, S, k, seed):
    from sluice_amd import ops

    rng = np.random.default_rng(seed)
    x = _bf16(rng.standard_normal((T, H)))
    q13 = torch.from_numpy(rng.standard_normal((S, 2 * I, H)).astype(np.float32) * 0.5).to(
        torch.float8_e4m3fn).view(torch.uint8)
    q2 = torch.from_numpy(rng.standard_normal((S, H, I)).astype(np.float32) * 0.5).to(
        torch.float8_e4m3fn).view(torch.uint8)
    s13 = (rng.random((S, 2 * I // 128, H // 128)) * 0.02 + 0.01).astype(np.float32)
    s2 = (rng.random((S, H // 128, I // 128)) * 0.02 + 0.01).astype(np.float32)
    ids = _routing(T, E, k, rng)
    tw = rng.random((T, k)).astype(np.float32)
    emap = _emap(E, S, rng, 0.9)
    out = ops.fused_experts(
        x.to(DEV), q13.to(DEV), q2.to(DEV), torch.from_numpy(tw).to(DEV),
        torch.from_numpy(ids).to(DEV), global_num_experts=E,
        expert_map=torch.from_numpy(emap).to(DEV), w1_scale=torch.from_numpy(s13).to(DEV),
        w2_scale=torch.from_numpy(s2).to(DEV), block_shape=[128, 128])
    torch.cuda.synchronize()
    w13f = om.dequant_block(q13.numpy(), s13)
    w2f = om.dequant_block(q2.numpy(), s2)
    ref = om.fused_experts(x.float().numpy(), w13f, w2f, tw, ids, expert_map=emap)
    return out.float().cpu().numpy(), ref


@pytest.mark.parametrize("T,H,I,E,S,k", [
    (8, 7168, 2048, 256, 6, 8),     # DeepSeek-V3 expert shape
    (1, 7168, 2048, 256, 4, 8),
    (12, 512, 256, 16, 8, 4),
    (80, 1152, 640, 48, 48, 4),     # the tiled kernels, 32-pair tiles
    (400, 1152, 640, 48, 48, 4),    # 64-pair tiles
])
def test_fused_experts_fp8(T, H, I, E, S, k):
    print(f"fused fp8 T={T} H={H} I={I} E={E} S={S} k={k}", flush=True)
    got, ref = _fp8_case(T, H, I, E, S, k, seed=T + I)
    err = om.rel_l2(got, ref)
    print(f"  rel_l2={err:.2e}", flush=True)
    assert err <= FP8_TOL


def test_fp8_decode_all_bytes_exact():
    """Every e4m3fn byte value decodes exactly: one expert whose gate row r
    holds byte r at column 0 (NaN encodings zeroed), up rows hold 1.0, the
    down projection is the identity, x = e_0 and all scales are 1, so
    out[r] = silu(decode(r)) up to the bf16 rounding of the result."""
    from sluice_amd import ops

    H = I = 256
    vals = np.arange(256, dtype=np.uint8)
    vals[vals == 0x7F] = 0
    vals[vals == 0xFF] = 0
    q13 = np.zeros((1, 2 * I, H), np.uint8)
    q13[0, :I, 0] = vals
    q13[0, I:, 0] = 0x38  # 1.0
    q2 = np.zeros((1, H, I), np.uint8)
    q2[0, np.arange(H), np.arange(I)] = 0x38
    s13 = np.ones((1, 2 * I // 128, H // 128), np.float32)
    s2 = np.ones((1, H // 128, I // 128), np.float32)
    x = torch.zeros((1, H), dtype=torch.bfloat16)
    x[0, 0] = 1.0
    out = ops.fused_experts(x.to(DEV), torch.from_numpy(q13).to(DEV), torch.from_numpy(q2).to(DEV),
                            torch.ones((1, 1), device=DEV),
                            torch.zeros((1, 1), dtype=torch.int32, device=DEV),
                            w1_scale=torch.from_numpy(s13).to(DEV),
                            w2_scale=torch.from_numpy(s2).to(DEV), block_shape=[128, 128])
    torch.cuda.synchronize()
    g = om.fp8_e4m3fn_to_f32(vals).astype(np.float64)
    want = g / (1 + np.exp(-g))
    got = out.float().cpu().numpy()[0]
    np.testing.assert_allclose(got, want, rtol=8e-3, atol=1e-30)


def _tile_case(T, H, I, Is, E, S, k, frac, fp8, seed):
    """Device inputs of a fused_experts call: (args, kwargs)."""
    rng = np.random.default_rng(seed)
    g = torch.Generator(device=DEV).manual_seed(seed)

    def weights(shape):
        w = torch.randn(shape, generator=g, device=DEV)
        if not fp8:
            return (w * 0.02).to(torch.bfloat16), None
        s = torch.rand((*shape[:-2], shape[-2] // 128, shape[-1] // 128), generator=g, device=DEV)
        return (w * 0.5).to(torch.float8_e4m3fn).view(torch.uint8), s * 0.02 + 0.01

    x = torch.randn((T, H), generator=g, device=DEV).to(torch.bfloat16)
    (w13, s13), (w2, s2) = weights((S, 2 * I, H)), weights((S, H, I))
    ids = _routing(T, E, k, rng)
    ids[T // 2] = E + 5  # out of range: the token's pairs are not resident
    tw = torch.from_numpy(rng.random((T, k)).astype(np.float32)).to(DEV)
    kw = dict(global_num_experts=E, routed_scaling_factor=1.5,
              expert_map=torch.from_numpy(_emap(E, S, rng, frac)).to(DEV))
    if fp8:
        kw.update(w1_scale=s13, w2_scale=s2, block_shape=[128, 128])
    if Is:
        (kw["shared_w1"], a), (kw["shared_w2"], b) = weights((2 * Is, H)), weights((H, Is))
        if fp8:
            kw.update(shared_w1_scale=a, shared_w2_scale=b)
    return [x, w13, w2, tw, torch.from_numpy(ids).to(DEV)], kw


def _in_slices(args, kw, n):
    """The call in slices of n tokens (the decode kernels, for small n)."""
    from sluice_amd import ops

    x, w13, w2, tw, ids = args
    return torch.cat([ops.fused_experts(x[t:t + n], w13, w2, tw[t:t + n], ids[t:t + n], **kw)
                      for t in range(0, x.shape[0], n)])


@pytest.mark.parametrize("T,H,I,Is,E,S,k,frac,fp8", [
    (112, 1088, 448, 448, 40, 40, 5, 0.8, False),   # 14 pairs per expert: the smallest, odd sizes
    (111, 1088, 448, 448, 40, 40, 5, 0.8, False),   # below the line
    (257, 1088, 448, 896, 64, 40, 5, 0.8, False),   # 64-pair tiles, partial ones
    (801, 2112, 1472, 0, 40, 40, 5, 1.0, False),    # 128-pair tiles
    (1000, 1088, 448, 448, 40, 40, 5, 0.8, False),  # over 4096 pairs: one prefill call
    (900, 64, 64, 0, 512, 512, 8, 0.9, False),      # over 4096 pairs, few per slot, one K chunk
    (600, 64, 64, 0, 512, 512, 8, 0.9, False),      # below the line in one call
    (301, 2048, 1024, 0, 16, 16, 16, 1.0, False),   # every token to every expert
    (300, 1088, 448, 448, 64, 40, 5, 0.0, False),   # nothing routed is resident
    (72, 1152, 640, 640, 48, 48, 4, 0.8, True),     # fp8, 32-pair tiles: the smallest
    (500, 1152, 640, 640, 48, 48, 4, 1.0, True),    # fp8, 64-pair tiles
    (1100, 1152, 640, 0, 64, 48, 4, 0.8, True),     # fp8, over 4096 pairs
    (96, 9216, 1024, 0, 40, 32, 4, 1.0, True),      # over 64 scale chunks of K
    (1700, 512, 256, 0, 64, 64, 5, 1.0, False),     # over 8192 pairs: the sort's next form
    (4200, 64, 64, 0, 64, 64, 8, 0.9, False),       # over 32768 pairs: its largest
])
def test_tiled_product_matches_the_decode_kernels(T, H, I, Is, E, S, k, frac, fp8):
    """Bit for bit: a token's output does not depend on how many others its
    call holds."""
    from sluice_amd import ops

    print(f"tiles T={T} H={H} I={I} Is={Is} E={E} S={S} k={k} fp8={fp8}", flush=True)
    args, kw = _tile_case(T, H, I, Is, E, S, k, frac, fp8, seed=T + H)
    got = [ops.fused_experts(*args, **kw) for _ in range(2)]
    ref = _in_slices(args, kw, 7)
    torch.cuda.synchronize()
    assert torch.equal(got[0], got[1])
    assert torch.equal(got[0], ref)


@pytest.mark.parametrize("fp8", [False, True])
def test_tiled_product_does_not_depend_on_the_slots(fp8):
    """The same experts in other slots give the same bits."""
    from sluice_amd import ops

    args, kw = _tile_case(300, 1152, 640, 0, 40, 24, 5, 1.0, fp8, seed=12)
    want = ops.fused_experts(*args, **kw)
    perm = torch.randperm(24, generator=torch.Generator().manual_seed(1)).to(DEV)
    inv = torch.empty_like(perm)
    inv[perm] = torch.arange(24, device=DEV)
    moved = [args[0], args[1][perm], args[2][perm], *args[3:]]
    emap = kw["expert_map"].long()
    kw["expert_map"] = torch.where(emap >= 0, inv[emap.clamp(min=0)], emap).to(torch.int32)
    for n in ("w1_scale", "w2_scale"):
        if n in kw:
            kw[n] = kw[n][perm]
    got = ops.fused_experts(*moved, **kw)
    torch.cuda.synchronize()
    assert (want != 0).any()
    assert torch.equal(got, want)


def _kernels(call):
    """Names of the kernels that call() launches."""
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        call()
        torch.cuda.synchronize()
    return " ".join(e.key for e in prof.key_averages())


@pytest.mark.parametrize("T,H,I,Is,E,S,k,fp8,route", [
    (10, 64, 1408, 2816, 64, 48, 6, False, "gemm1_self"),   # 7040 workgroups
    (11, 64, 1408, 2816, 64, 48, 6, False, "align"),        # 7744
    (16, 128, 256, 0, 16, 16, 6, True, "gemm1_self"),
    (17, 128, 256, 0, 16, 16, 5, True, "align"),            # a slot may have two blocks
    (111, 1088, 448, 448, 40, 40, 5, False, "align"),
    (112, 1088, 448, 448, 40, 40, 5, False, "tile"),        # 14 pairs per expert
    (178, 1088, 448, 0, 64, 40, 5, False, "align"),         # ... of all, resident or not
    (180, 1088, 448, 0, 64, 40, 5, False, "tile"),
    (71, 1152, 640, 640, 48, 48, 4, True, "align"),
    (72, 1152, 640, 640, 48, 48, 4, True, "tile"),          # 6, fp8
    (600, 64, 64, 0, 512, 512, 8, False, "align"),          # over 4096 pairs
    (900, 64, 64, 0, 512, 512, 8, False, "tile"),
])
def test_which_kernels_run(T, H, I, Is, E, S, k, fp8, route):
    """Both sides of each line: other kernels there were measured slower."""
    from sluice_amd import ops

    args, kw = _tile_case(T, H, I, Is, E, S, k, 1.0, fp8, seed=T)
    ops.fused_experts(*args, **kw)
    names = _kernels(lambda: ops.fused_experts(*args, **kw))
    ran = [r for r in ("gemm1_self", "align", "tile") if f"moe_{r}_kernel" in names]
    assert ran == [route], names


def test_tiled_product_keeps_tokens_apart():
    """A token of NaN and one of infinities change no other token's bits."""
    from sluice_amd import ops

    args, kw = _tile_case(257, 1088, 448, 448, 40, 40, 5, 1.0, False, seed=3)
    clean = ops.fused_experts(*args, **kw)
    args[0][13] = float("nan")
    args[0][200] = float("inf")
    got = ops.fused_experts(*args, **kw)
    torch.cuda.synchronize()
    assert torch.isnan(got[13]).any()
    rest = [t for t in range(257) if t not in (13, 200)]
    assert torch.equal(got[rest], clean[rest])


def test_prefill_entry_bounds():
    """Refused without touching the GPU: too many pairs, scales of one weight
    only, sizes the kernels do not take."""
    from sluice_amd import _lib

    lib = _lib.load()
    buf = torch.empty(1 << 20, dtype=torch.uint8, device=DEV)
    p = buf.data_ptr()

    def call(T, H, I, s13=None, s2=None, shared=None):
        return lib.sluice_fused_experts_prefill(
            p, p, s13, p, s2, p, p, None, T, H, I, 8, 64, 64, 1.0, shared, None, shared, None,
            I if shared else 0, None, p, buf.numel(), p, None)

    assert call(8193, 64, 64) == _lib.SLUICE_E_INVAL     # 65544 pairs
    assert call(8000, 64, 64, shared=p) == _lib.SLUICE_E_INVAL
    assert call(1024, 64, 64) == _lib.SLUICE_E_INVAL     # workspace too small
    assert call(8, 128, 128, s13=p) == _lib.SLUICE_E_INVAL
    assert call(8, 192, 128, s13=p, s2=p) == _lib.SLUICE_E_INVAL
    assert call(8, 96, 64) == _lib.SLUICE_E_INVAL


def test_prefill_slices_follow_the_reserved_workspace(monkeypatch):
    """While a graph is captured a chunk whose workspace was not reserved runs
    in slices that fit the one there is; the replays give the eager bits."""
    from sluice_amd import ops

    args, kw = _tile_case(1000, 1088, 448, 0, 40, 40, 5, 0.8, False, seed=5)
    want = ops.fused_experts(*args, **kw)
    monkeypatch.setattr(ops, "_WS", ops._Workspace())
    ops.reserve_workspace(DEV, 819, 1088, 448, 5)  # 4095 pairs
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = ops.fused_experts(*args, **kw)
    for _ in range(3):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)


def test_graphs_replay_after_a_longer_eager_call(monkeypatch):
    """A graph captured over the reserved workspace gives the eager bits after
    an eager call that needs more than it holds, with the memory that this
    call gave back written over."""
    from sluice_amd import ops

    args, kw = _tile_case(1000, 1088, 448, 0, 40, 40, 5, 0.8, False, seed=6)
    short = [args[0][:5], args[1], args[2], args[3][:5], args[4][:5]]
    monkeypatch.setattr(ops, "_WS", ops._Workspace())
    ops.reserve_workspace(DEV, 5, 1088, 448, 5)
    want, want_long = ops.fused_experts(*short, **kw), None
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = ops.fused_experts(*short, **kw)
    for i in range(3):
        long = ops.fused_experts(*args, **kw)
        over = [torch.full((n,), float("nan"), device=DEV) for n in (1 << 18, 1 << 23)]
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
        assert all(torch.isnan(t).all() for t in over)
        assert want_long is None or torch.equal(long, want_long)
        want_long = long
        ops.fused_experts(args[0][:700], args[1], args[2], args[3][:700], args[4][:700], **kw)


def test_tiled_product_over_a_map_whose_slots_streamed():
    """A prefill call over a layer's registered map, whose last gap filled
    slots (all landed by then: the layer's own product waited), gives the
    decode kernels' product.  Rows in flight: test_gpu_gap.py."""
    from sluice_amd import ops
    from sluice_amd.decoder import SyntheticMoELayer, build_offloaded

    E, S, k, H, I = 24, 16, 4, 2048, 1024
    layer = SyntheticMoELayer(H, I, E, k, renorm=True, seed=4, device=DEV)
    off = build_offloaded([layer], slots=S, device=DEV)
    try:
        g = torch.Generator(device=DEV).manual_seed(6)
        layer(torch.randn((4, H), generator=g, device=DEV).to(torch.bfloat16))  # fills slots
        x = torch.randn((96, H), generator=g, device=DEV).to(torch.bfloat16)
        ids = torch.randint(0, E, (96, k), generator=g, device=DEV, dtype=torch.int32)
        tw = torch.rand((96, k), generator=g, device=DEV)
        args = [x, layer.w13_weight, layer.w2_weight, tw, ids]
        kw = dict(global_num_experts=E, expert_map=layer.expert_map)
        got = ops.fused_experts(*args, **kw)
        ref = _in_slices(args, kw, 4)
        torch.cuda.synchronize()
        assert (ref != 0).any()
        assert torch.equal(got, ref)
    finally:
        off.close()


def test_fused_experts_goes_through_the_op_when_something_watches():
    """A dispatch mode, the profiler and autograd see the op; a plain eager
    call gives its bits without it; make_fx and vmap-free tracing get one node."""
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.utils._python_dispatch import TorchDispatchMode

    from sluice_amd import ops

    args, kw = _tile_case(3, 256, 64, 64, 8, 8, 2, 1.0, False, seed=8)
    want = torch.ops.sluice.fused_experts(*args, **kw)
    assert torch.equal(ops.fused_experts(*args, **kw), want)
    seen = []

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, a=(), k=None):
            seen.append(str(func))
            return func(*a, **(k or {}))

    with Watch():
        assert torch.equal(ops.fused_experts(*args, **kw), want)
    assert any("fused_experts" in s for s in seen)
    g = make_fx(lambda x: ops.fused_experts(x, *args[1:], **kw))(args[0])
    assert any("fused_experts" in str(n.target) for n in g.graph.nodes)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        ops.fused_experts(*args, **kw)
    assert any("fused_experts" in e.key for e in prof.key_averages())
    x = args[0].clone().requires_grad_()
    assert ops.fused_experts(x, *args[1:], **kw).requires_grad == torch.ops.sluice.fused_experts(
        x, *args[1:], **kw).requires_grad
    with pytest.raises(TypeError):
        ops.fused_experts(*args, **kw, no_such_argument=1)


def test_function_modes_and_lazy_views_go_through_the_op():
    """A torch-function mode sees the op; routing weights that are lazily
    negated or lazily zero have their values."""
    from torch.overrides import TorchFunctionMode

    from sluice_amd import ops

    args, kw = _tile_case(3, 256, 64, 0, 8, 8, 2, 1.0, False, seed=8)
    want = torch.ops.sluice.fused_experts(*args, **kw)
    seen = []

    class Watch(TorchFunctionMode):
        def __torch_function__(self, func, types, a=(), k=None):
            seen.append(str(func))
            return func(*a, **(k or {}))

    with Watch():
        assert torch.equal(ops.fused_experts(*args, **kw), want)
    assert any("fused_experts" in s for s in seen)
    tw = args[3]
    neg = torch.complex(tw, -tw).conj().imag
    assert neg.is_neg() and torch.equal(neg, tw)
    args[3] = neg
    assert torch.equal(ops.fused_experts(*args, **kw), want)
    args[3] = torch._efficientzerotensor(tw.shape, dtype=tw.dtype, device=DEV)
    assert (ops.fused_experts(*args, **kw) == 0).all()


@pytest.mark.parametrize("T,k,E,S,how", [
    (1, 1, 1, 1, "even"),          # one pair
    (1, 6, 64, 48, "even"),
    (12, 8, 128, 96, "even"),      # 96 pairs: the largest call that plans itself
    (97, 1, 64, 64, "even"),       # the align launch
    (31, 3, 4, 4, "even"),         # about 23 pairs per slot: a block and a rest
    (48, 2, 16, 16, "one"),        # every pair to one expert: six full blocks
    (9, 8, 512, 512, "even"),
    (9, 4, 16, 8, "outside"),      # no pair is resident
    (12, 8, 16, 16, "one"),        # 96 pairs of 12 tokens to one expert: six blocks
    (16, 6, 16, 16, "even"),
    (17, 5, 16, 16, "even"),       # more tokens than a block: the align launch
])
@pytest.mark.parametrize("fp8", [False, True])
def test_small_calls_plan_themselves(T, k, E, S, how, fp8):
    """Without a plan a small call groups its pairs in gemm1; the bits are
    those of the stages run over an align plan."""
    from sluice_amd import _lib, ops

    H, I = 256, 128
    args, kw = _tile_case(T, H, I, 0, E, S, k, 0.9 if S < E else 1.0, fp8, seed=T + E) \
        if T > 1 else _tile_case(2, H, I, 0, E, S, k, 1.0, fp8, seed=E)
    x, w13, w2, tw, ids = args
    x, tw, ids = x[:T].contiguous(), tw[:T].contiguous(), ids[:T].contiguous()
    if how == "one":
        ids[:] = 3
    elif how == "outside":
        ids[:] = -1
    kw["routed_scaling_factor"] = 1.0
    st = torch.cuda.current_stream().cuda_stream
    ref = _staged(_lib.load(), x, w13, w2, tw, ids, kw["expert_map"], T, H, I, E, S, k, 1.0, None,
                  st, fp8=(kw["w1_scale"], kw["w2_scale"]) if fp8 else None)
    for _ in range(3):
        got = ops.fused_experts(x, w13, w2, tw, ids, **kw)
        torch.cuda.synchronize()
        assert torch.equal(got, ref)
    if how != "outside":
        assert (ref != 0).any()
