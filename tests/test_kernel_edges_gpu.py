"""The kernels' tile edges, remainders and dispatch rules against the CPU oracle."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from wisp import kernels, quant

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("bits", [8, 4, 3, 2])
@pytest.mark.parametrize("n", [128, 17 * 128, 16 * 128])  # 3, 51 and 48 groups: part of a workgroup, a remainder, whole ones
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shift", [0, 1])  # 1: values that are not 16-byte aligned take the general kernel
def test_quantize_group_128_edges(bits, n, dtype, shift):
    rng = np.random.default_rng(bits + n)
    w = (rng.standard_normal(3 * n) * 0.05).astype(np.float32)
    w[:128] = rng.integers(0, 2 * 2**bits - 1, 128) * np.float32(0.5)  # quotients at and next to ties
    w[128:256] *= np.float32(1e-4)  # scale clamped to 1e-5, an fp16 subnormal
    w[256:384] *= np.float32(3e6)  # minimum beyond fp16: -inf, and infinite quotients
    w = O.bf16_bits_to_f32(O.f32_to_bf16_bits(w)) if dtype == torch.bfloat16 else w
    buf = torch.zeros(3 * n + shift, dtype=dtype, device=DEV)
    buf[shift:] = torch.from_numpy(w).to(DEV)
    got = quant.quantize(buf[shift:].view(3, n), bits, 128).cpu().numpy()
    assert np.array_equal(got, O.quantize(w, bits, 128))


# capacities past 128 chunks of 64 positions merge with eight waves per head: the first 64 chunks by the lower four,
# the rest by all of them, in batches of 16 per wave
@pytest.mark.parametrize("Hq,Hk,D", [(8, 2, 128), (4, 2, 64), (2, 2, 256)])
def test_attn_decode_wide_merge(Hq, Hk, D):
    T = 128 * 64 + 64 * 70  # 198 chunks: 64, then 8 x 16, then 6
    gen = torch.Generator(device=DEV).manual_seed(Hq + D)
    q, k, v = (torch.randn(s, generator=gen, device=DEV).to(torch.bfloat16)
               for s in ((1, Hq, 1, D), (1, Hk, T, D), (1, Hk, T, D)))
    for pos in (0, 63, 64, 4095, 4096, 4159, 8191, 12287, 12288, T - 1):
        p = torch.tensor([pos], device=DEV)
        kn, vn = k.clone(), v.clone()
        kn[:, :, pos + 1 :], vn[:, :, pos + 1 :] = float("nan"), float("nan")  # nothing past the position is read
        got = kernels.attn_decode(q, kn, vn, p, D**-0.5).view(Hq, D).double()
        kk = k[0, :, : pos + 1].double().repeat_interleave(Hq // Hk, 0)
        vv = v[0, :, : pos + 1].double().repeat_interleave(Hq // Hk, 0)
        w = ((kk @ q[0, :, 0].double()[:, :, None])[..., 0] * D**-0.5).softmax(-1)
        ref = (w[:, None] @ vv)[:, 0]
        # one bf16 rounding (2^-9 of a value at most) and fp32 sums
        assert ((got - ref).norm() / ref.norm()).item() <= 2.0**-8, pos


# kernel 1 rows of 2, 3 and 4 chunks per lane (a remainder in each; float32 x of four goes to the generic kernel),
# kernel 2 with 4 to 512 (expert, chunk) pairs: part of one step, every step count, and more than 16 experts
@pytest.mark.parametrize("bits", [4, 3, 2])
@pytest.mark.parametrize("H,I,group,k", [(2176, 128, 128, 1), (4096, 256, 256, 3), (4224, 128, 128, 17), (6272, 128, 128, 2),
                                         (8192, 128, 128, 2), (256, 640, 128, 5), (4096, 512, 256, 13), (256, 1152, 128, 6),
                                         (128, 1408, 128, 10), (128, 8192, 128, 2), (512, 384, 128, 16)])
def test_wide_decode_layers(bits, H, I, group, k):
    rng = np.random.default_rng(H + I + k + bits)
    n, E = H * I, k + 1
    pool = np.stack([O.quantize((rng.standard_normal(3 * n) * 0.02).astype(np.float32), bits, group) for _ in range(E)])
    slots, w = rng.permutation(E)[:k], rng.random(k).astype(np.float32)
    pt = torch.from_numpy(pool).to(DEV)
    meta = torch.from_numpy(O.meta(slots, w)).to(DEV)
    for xdt, tol in ((torch.bfloat16, 2.0**-8), (torch.float32, 4e-6)):  # one rounding of the result; fp32 sums
        x = torch.from_numpy(rng.standard_normal(H).astype(np.float32)).to(xdt)
        _, _, ref = O.moe_layer_f64(pool, slots, w, x.float().numpy(), H, I, bits, group)
        got = kernels.moe_decode_fast(pt, meta, x.to(DEV), k, n, H, I, bits, group).double().cpu().numpy()
        err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
        print(f"H={H} I={I} k={k} bits={bits} {xdt}: {err:.2e}")
        assert err <= tol
    bad = meta.clone()
    bad[k - 1] = E  # not a slot: NaN, nothing read
    assert torch.isnan(kernels.moe_decode_fast(pt, bad, x.to(DEV), k, n, H, I, bits, group)).all()
