"""The kernels' tile edges, remainders and dispatch rules against the CPU oracle."""
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from oracle import oracle as O
from wisp import _lib, kernels, quant
from wisp.cache import ExpertCache
from wisp.moe import PagedMoEBlock, Runtime, route
from wisp.store import ExpertStore

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


# units of 8 values, 1,024 per workgroup: part of one, whole ones, a remainder; groups of 2^i take the unit kernel, 96 not
@pytest.mark.parametrize("bits", [8, 4, 3, 2])
@pytest.mark.parametrize("n,group", [(32, 32), (128, 128), (8192, 64), (8192 + 256, 256), (4096 * 3 + 32, 32), (960, 96)])
def test_dequant_unit_edges(bits, n, group):
    rng = np.random.default_rng(bits * n + group)
    w = (rng.standard_normal((3, 3 * n)) * 0.05).astype(np.float32)
    w[1, :group] *= np.float32(1e-4)  # a scale that is an fp16 subnormal
    rows = np.stack([O.quantize(v, bits, group) for v in w])
    pad = -rows.shape[1] % 16
    pool = torch.from_numpy(np.pad(rows, ((0, 0), (0, pad)), constant_values=0xA5)).to(DEV)
    idx = [2, 0, 1, 2, 3, -1]
    got = quant.dequant_rows(pool, torch.tensor(idx, device=DEV), n, bits, group).view(torch.int16).cpu().numpy().view(np.uint16)
    ref = O.dequant(rows, n, bits, group).reshape(3, 3, n)
    for g, i in zip(got, idx):
        if 0 <= i < 3:
            assert np.array_equal(g, ref[i])
        else:
            assert (g == 0x7FC0).all()


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


# a short context in a large cache merges as in a small one, bit for bit: up to 128 chunks by four waves
@pytest.mark.parametrize("Hq,Hk,D", [(8, 2, 128), (4, 2, 64), (2, 2, 256)])
def test_attn_decode_short_context_in_a_large_cache(Hq, Hk, D):
    gen = torch.Generator(device=DEV).manual_seed(Hq + D)
    q, k, v = (torch.randn(s, generator=gen, device=DEV).to(torch.bfloat16)
               for s in ((1, Hq, 1, D), (1, Hk, 8192 + 64, D), (1, Hk, 8192 + 64, D)))
    ks, vs = k[:, :, :8192].contiguous(), v[:, :, :8192].contiguous()
    for pos in (0, 64, 4031, 4095, 4096, 4160, 8127, 8128, 8191):
        p = torch.tensor([pos], device=DEV)
        got, want = kernels.attn_decode(q, k, v, p, D**-0.5), kernels.attn_decode(q, ks, vs, p, D**-0.5)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), pos
    # one chunk more: all eight waves
    got = kernels.attn_decode(q, k, v, torch.tensor([8192], device=DEV), D**-0.5).view(Hq, D).double()
    kk, vv = (t[0, :, :8193].double().repeat_interleave(Hq // Hk, 0) for t in (k, v))
    w = ((kk @ q[0, :, 0].double()[:, :, None])[..., 0] * D**-0.5).softmax(-1)
    ref = (w[:, None] @ vv)[:, 0]
    assert ((got - ref).norm() / ref.norm()).item() <= 2.0**-8  # one bf16 rounding and fp32 sums


# kernel 1 rows of 2, 3 and 4 chunks per lane (a remainder in each; float32 x of four, or of few rows, goes to the generic
# kernel), kernel 2 with 4 to 512 (expert, chunk) pairs and more than 16 experts, whichever kernel the rules give them
# (the next test has every form of the wide ones)
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


def _group_64(rows, n, bits):
    """The same weights with every group of 128 as two of 64 that share its scale and minimum."""
    nc, ng = 3 * n * bits // 8, 3 * n // 128
    fp16 = rows[:, nc : nc + 4 * ng].copy().view(np.uint16)
    return np.concatenate([rows[:, :nc], np.repeat(fp16, 2, axis=1).view(np.uint8)], axis=1)


# the kernels for long rows and for any (expert, chunk) count against the general ones, which take groups of 64: the same
# bits, a weighted sum of whole experts also where a routing weight is not finite. k_down's order of the sums (16, 8, 4, 2
# and 1 lanes per sum, k <= 16) and k_down_generic's (more experts, more chunks than a wave, more LDS than it takes)
@pytest.mark.parametrize("bits", [4, 3, 2])
@pytest.mark.parametrize("H,I,k", [(4096, 1536, 8), (2176, 128, 1), (4224, 256, 17), (6272, 128, 2), (8192, 128, 2),
                                   (384, 1152, 5), (384, 1024, 3), (384, 640, 9), (384, 512, 16), (640, 384, 16),
                                   (384, 128, 65), (384, 8192, 2), (384, 2304, 7), (5120, 1408, 10), (4096, 1536, 4),
                                   (4096, 1280, 6), (4096, 1152, 10), (3072, 1152, 10), (4096, 1536, 10), (384, 1536, 4),
                                   (2176, 896, 2), (4096, 256, 8), (4096, 640, 3), (3072, 1792, 7), (4096, 384, 40), (384, 128, 17),
                                   (384, 128, 40), (384, 128, 60), (4096, 128, 60), (4096, 128, 90)])
def test_wide_decode_layers_equal_the_general_kernels(bits, H, I, k):
    rng = np.random.default_rng(H + I + k + bits)
    n, E = H * I, k + 1
    some = np.stack([O.quantize((rng.standard_normal(3 * n) * 0.02).astype(np.float32), bits, 128) for _ in range(min(E, 4))])
    rows = some[np.arange(E) % len(some)]
    p128, p64 = torch.from_numpy(rows).to(DEV), torch.from_numpy(_group_64(rows, n, bits)).to(DEV)
    slots, w = rng.permutation(E)[:k], rng.random(k).astype(np.float32)
    for last in (w[-1], np.float32("inf"), np.float32("-inf"), np.float32("nan")):
        w[-1] = last
        meta = torch.from_numpy(O.meta(slots, w)).to(DEV)
        for xdt in (torch.bfloat16, torch.float16, torch.float32):
            x = torch.from_numpy(rng.standard_normal(H).astype(np.float32)).to(xdt).to(DEV)
            got = kernels.moe_decode_fast(p128, meta, x, k, n, H, I, bits, 128)
            want = kernels.moe_decode_fast(p64, meta, x, k, n, H, I, bits, 64)
            same = (got == want) | (torch.isnan(got) & torch.isnan(want))
            assert same.all(), (xdt, last, (~same).sum().item(), "of", H)
            assert torch.isfinite(got).all() if np.isfinite(last) else not torch.isfinite(got).any()
            if np.isinf(last):
                assert torch.isinf(got).all()


def _routing(gen, T, E, k):
    p = torch.randn((T, E), generator=gen, device=DEV).softmax(-1)
    rw, sel = p.topk(k, -1)
    return sel, rw.to(torch.bfloat16)


# the plan formed on the GPU against the host's, bit for bit: one token, runs that are not whole waves, every chunk size, the largest table, k = 32 (the wide combine)
@pytest.mark.parametrize("E,k,T,bits", [(6, 2, 1, 4), (6, 2, 17, 3), (4, 2, 900, 4), (300, 8, 50, 2), (512, 4, 40, 4),
                                        (40, 32, 33, 4), (3, 1, 9000, 4), (5, 3, 333, 3)])
@pytest.mark.parametrize("mode", ["all", "part", "twice", "outside"])
def test_prefill_plan_on_the_gpu_equals_the_hosts(E, k, T, bits, mode):
    H, I, n = 256, 128, 256 * 128
    rng = np.random.default_rng(E + T)
    pool = torch.from_numpy(np.stack([O.quantize((rng.standard_normal(3 * n) * 0.05).astype(np.float32), bits, 128)
                                      for _ in range(6)])).to(DEV)
    gen = torch.Generator(device=DEV).manual_seed(E * 31 + T)
    x = torch.randn((T, H), generator=gen, device=DEV).to(torch.bfloat16)
    sel, rw = _routing(gen, T, E, k)
    slots = {e: e % 6 for e in range(E)}
    if mode == "part":  # some experts absent, one with no such slot (its tokens become NaN)
        slots = {e: e % 6 for e in range(0, E, 2)}
        slots[max(slots)] = 77
    if mode == "twice":  # an expert chosen twice by one token
        sel[:, -1] = sel[:, 0]
    if mode == "outside":  # ids that no table holds
        sel[::3, 0], sel[1::3, -1] = -1, 1 << 40
    for w in (rw, rw.float(), rw.half()):
        got = kernels.moe_prefill(pool, slots, x, sel, w, n, H, I, bits)
        want = kernels.moe_prefill(pool, slots, x, sel.cpu(), w, n, H, I, bits)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    s32 = sel.clamp(max=1 << 20).int()
    acc, ref = torch.full((T, H), 0.25, device=DEV), torch.full((T, H), 0.25, device=DEV)
    kernels.moe_prefill(pool, slots, x, s32, rw, n, H, I, bits, acc=acc)
    kernels.moe_prefill(pool, slots, x, s32.cpu(), rw, n, H, I, bits, acc=ref)
    assert torch.equal(acc.view(torch.int32), ref.view(torch.int32))


# skewed routing, and the item sizes of a card that the experts' rows fill (by the parity of I / 128 and the width) and of
# one that they do not: the outputs do not depend on them
@pytest.mark.parametrize("bits", [4, 2])
@pytest.mark.parametrize("E,I,T", [(400, 128, 100), (400, 128, 700), (200, 256, 60), (200, 256, 500), (40, 256, 300)])
def test_prefill_plan_of_skewed_routing(bits, E, I, T):
    H, k, n = 256, 4, 256 * I
    rng = np.random.default_rng(E + T + bits)
    pool = torch.from_numpy(np.stack([O.quantize((rng.standard_normal(3 * n) * 0.05).astype(np.float32), bits, 128)
                                      for _ in range(5)])).to(DEV)
    key = -1.1 * np.log(np.arange(1, E + 1)) + rng.gumbel(size=(T, E))  # k different experts of a Zipf(1.1) draw
    sel = torch.from_numpy(rng.permutation(E)[np.argsort(-key, 1)[:, :k]].astype(np.int64))
    x = torch.from_numpy(rng.standard_normal((T, H)).astype(np.float32)).to(torch.bfloat16).to(DEV)
    rw = torch.from_numpy(rng.random((T, k)).astype(np.float32)).to(DEV)
    slots = {e: e % 5 for e in range(E)}
    got = kernels.moe_prefill(pool, slots, x, sel.to(DEV), rw, n, H, I, bits)
    want = kernels.moe_prefill(pool, slots, x, sel, rw, n, H, I, bits)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


# a hot expert has more matches in a wave's run of the pairs than its list of 256 holds: they are read again and placed by
# their ranks. Runs of 576 pairs (the last one partial) and of 1,088; all pairs of one expert, most, and two such experts
@pytest.mark.parametrize("T,k", [(9000, 1), (8640 + 33, 2), (8191, 1)])
@pytest.mark.parametrize("share", [1.0, 0.9, 0.5])
def test_prefill_plan_of_a_hot_expert(T, k, share):
    E, H, I, bits, n = 5, 256, 128, 4, 256 * 128
    rng = np.random.default_rng(T + k)
    pool = torch.from_numpy(np.stack([O.quantize((rng.standard_normal(3 * n) * 0.05).astype(np.float32), bits, 128)
                                      for _ in range(E)])).to(DEV)
    hot = rng.random(T) < share
    sel = np.stack([np.where(hot, 3, 1), np.where(hot, rng.integers(4, 6, T), 0)], 1)[:, :k]  # 5: an absent expert
    x = torch.from_numpy(rng.standard_normal((T, H)).astype(np.float32)).to(torch.bfloat16).to(DEV)
    rw = torch.from_numpy(rng.random((T, k)).astype(np.float32)).to(DEV)
    st = torch.from_numpy(np.ascontiguousarray(sel))
    slots = {e: (e + 2) % E for e in range(E)}
    got = kernels.moe_prefill(pool, slots, x, st.to(DEV), rw, n, H, I, bits)
    want = kernels.moe_prefill(pool, slots, x, st, rw, n, H, I, bits)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


def test_prefill_is_planned_on_the_host_where_the_workspace_does_not_fit(monkeypatch):
    """The GPU plan's workspace has room for all T * k pairs: a call that runs few of them must not need it."""
    E, k, T, H, I, bits, n = 8, 2, 70, 256, 128, 4, 256 * 128
    rng = np.random.default_rng(6)
    pool = torch.from_numpy(np.stack([O.quantize((rng.standard_normal(3 * n) * 0.05).astype(np.float32), bits, 128)
                                      for _ in range(E)])).to(DEV)
    gen = torch.Generator(device=DEV).manual_seed(10)
    x = torch.randn((T, H), generator=gen, device=DEV).to(torch.bfloat16)
    sel, rw = _routing(gen, T, E, k)
    for slots in ({1: 1, 6: 6}, {1: -(1 << 31), 6: 6}):  # and a slot that is the table's mark of an absent expert
        want = kernels.moe_prefill(pool, slots, x, sel.cpu(), rw, n, H, I, bits)
        assert torch.equal(kernels.moe_prefill(pool, slots, x, sel, rw, n, H, I, bits).view(torch.int16),
                           want.view(torch.int16))
        with monkeypatch.context() as m:
            m.setattr(kernels, "_plan_workspace", lambda nbytes, dev: None)
            got = kernels.moe_prefill(pool, slots, x, sel, rw, n, H, I, bits)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("on", ["cpu", DEV])
def test_prefill_of_a_width_without_kernels_where_no_pair_runs(on):
    """A call none of whose pairs has an expert is zeros, whatever its width: nothing is launched for it."""
    H, I, n = 256, 128, 256 * 128
    pool = torch.zeros((2, quant.expert_nbytes(n, 8, 128)), dtype=torch.uint8, device=DEV)
    x = torch.ones((3, H), dtype=torch.bfloat16, device=DEV)
    sel, rw = torch.full((3, 2), 9, device=on), torch.ones((3, 2), device=DEV)
    assert (kernels.moe_prefill(pool, {0: 0, 1: 1}, x, sel, rw, n, H, I, 8) == 0).all()
    with pytest.raises(ValueError):
        kernels.moe_prefill(pool, {9: 0}, x, sel, rw, n, H, I, 8)


def test_prefill_under_graph_capture_follows_the_routing():
    E, k, T, H, I, bits, n = 8, 2, 70, 256, 128, 4, 256 * 128
    rng = np.random.default_rng(5)
    pool = torch.from_numpy(np.stack([O.quantize((rng.standard_normal(3 * n) * 0.05).astype(np.float32), bits, 128)
                                      for _ in range(E)])).to(DEV)
    gen = torch.Generator(device=DEV).manual_seed(9)
    x = torch.randn((T, H), generator=gen, device=DEV).to(torch.bfloat16)
    sel, rw = _routing(gen, T, E, k)
    slots = {e: e for e in range(E)}
    kernels.moe_prefill(pool, slots, x, sel, rw, n, H, I, bits)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = kernels.moe_prefill(pool, slots, x, sel, rw, n, H, I, bits)
    for _ in range(4):
        s2, r2 = _routing(gen, T, E, k)
        sel.copy_(s2)
        rw.copy_(r2)
        g.replay()
        torch.cuda.synchronize()
        want = kernels.moe_prefill(pool, slots, x, s2.cpu(), r2, n, H, I, bits)
        assert torch.equal(out.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("nslots,n_static,policy", [(12, 0, "lru"), (16, 3, "lru"), (9, 0, "lru"), (12, 0, "wsa")])
def test_block_runs_all_experts_at_once_where_the_cache_holds_them(nslots, n_static, policy):
    """A paged block's prefill pages in chunks of rt.chunk experts whatever the cache holds: the bookkeeping equals the
    chunk-by-chunk calls, and the output the oracle's, with and without room for all routed experts."""
    E, k, T, H, I, bits, n = 12, 4, 40, 256, 128, 4, 256 * 128
    gen = torch.Generator(device=DEV).manual_seed(nslots + n_static)
    store = ExpertStore(1, E, n, bits, 128)
    store.fill(((e, torch.randn((3, n), generator=gen, device=DEV) * 0.05) for e in range(E)))
    pre = list(range(n_static))
    caches = [ExpertCache(store, nslots, policy=policy, n_static=n_static, preload_keys=pre or None) for _ in range(2)]
    rt = Runtime(store, caches[0], chunk=5)
    gate = torch.nn.Linear(H, E, bias=False, device=DEV, dtype=torch.bfloat16)
    cfg = SimpleNamespace(hidden_size=H, moe_intermediate_size=I, num_experts=E, num_experts_per_tok=k,
                          norm_topk_prob=True)
    block = PagedMoEBlock(gate, 0, rt, cfg)
    for step in range(3):
        x = torch.randn((1, T, H), generator=gen, device=DEV).to(torch.bfloat16)
        with torch.no_grad():
            y = block(x)
            logits = gate(x[0])
        y = y[0] if isinstance(y, tuple) else y
        sel, rw = route(logits, k, True, x.dtype)
        keys = torch.unique(sel.cpu()).tolist()
        want = []
        for i in range(0, len(keys), 5):
            want += list(zip(keys[i : i + 5], caches[1].ensure(keys[i : i + 5])))
        a, b = caches[0].core, caches[1].core
        assert a.stats == b.stats
        assert [a.lookup(e) for e in range(E)] == [b.lookup(e) for e in range(E)]
        xb = x[0].view(torch.int16).cpu().numpy().view(np.uint16)
        ref = O.moe_prefill_f64(store.host.numpy(), {e: e for e in range(E)}, xb, sel.cpu().numpy(),
                                rw.float().cpu().numpy(), H, I, bits)
        err = np.linalg.norm(y[0].double().cpu().numpy() - ref) / np.linalg.norm(ref)
        assert err <= 2.0**-8, (step, err)
    for c in caches:
        c.free()


def test_block_pages_in_chunks_where_the_workspace_for_all_pairs_does_not_fit(monkeypatch):
    """Memory that holds a chunk's workspace but not the one for all pairs: the block's prefill runs chunk by chunk, with
    the bits and the bookkeeping of a block whose cache does not hold all experts at once."""
    E, k, T, H, I, bits, n = 12, 4, 40, 256, 128, 4, 256 * 128
    gen = torch.Generator(device=DEV).manual_seed(21)
    store = ExpertStore(1, E, n, bits, 128)
    store.fill(((e, torch.randn((3, n), generator=gen, device=DEV) * 0.05) for e in range(E)))
    caches = [ExpertCache(store, E, policy="lru") for _ in range(2)]
    gate = torch.nn.Linear(H, E, bias=False, device=DEV, dtype=torch.bfloat16)
    cfg = SimpleNamespace(hidden_size=H, moe_intermediate_size=I, num_experts=E, num_experts_per_tok=k,
                          norm_topk_prob=True)
    blocks = [PagedMoEBlock(gate, 0, Runtime(store, c, chunk=5), cfg) for c in caches]
    monkeypatch.setattr(caches[1], "holds_at_once", lambda n: False)
    most, empty = _lib.lib().wisp_prefill_ws_bytes(T * k, H, I), torch.empty

    def small(size, *a, **kw):
        if kw.get("dtype") == torch.uint8 and size >= most:
            raise torch.OutOfMemoryError("refused by the test")
        return empty(size, *a, **kw)

    for _ in range(2):
        x = torch.randn((1, T, H), generator=gen, device=DEV).to(torch.bfloat16)
        got = []
        for refuse, block in ((True, blocks[0]), (False, blocks[1])):
            with torch.no_grad(), monkeypatch.context() as m:
                if refuse:
                    m.setattr(kernels.torch, "empty", small)
                y = block(x)
            got.append(y[0] if isinstance(y, tuple) else y)
        assert torch.equal(got[0].view(torch.int16), got[1].view(torch.int16))
        a, b = caches[0].core, caches[1].core
        assert a.stats == b.stats
        assert [a.lookup(e) for e in range(E)] == [b.lookup(e) for e in range(E)]
        assert blocks[0].rt.stats == blocks[1].rt.stats
    for c in caches:
        c.free()


# the LDS-DMA GEMMs at every code width: one and several steps, more than 16 K groups, passes of 1 to 8 token tiles and
# several of them, and an odd number of K groups in the down projection (its register form beside them)
@pytest.mark.parametrize("bits", [4, 3, 2])
@pytest.mark.parametrize("E,H,I,T,k", [(3, 256, 256, 2, 1), (4, 512, 512, 90, 2), (3, 4352, 256, 20, 2), (2, 256, 2304, 40, 1),
                                       (2, 256, 2176, 30, 2), (3, 256, 384, 200, 2), (2, 1024, 256, 300, 2)])
def test_prefill_dma_every_width(bits, E, H, I, T, k):
    n = H * I
    rng = np.random.default_rng(E * H + I + T + bits)
    pool = np.stack([O.quantize((rng.standard_normal(3 * n) * 0.03).astype(np.float32), bits, 128) for _ in range(E)])
    sel, rw = O.route(rng.standard_normal((T, E)).astype(np.float32), k)
    x = O.f32_to_bf16_bits(rng.standard_normal((T, H)).astype(np.float32)).reshape(T, H)
    ref = O.moe_prefill_f64(pool, {e: e for e in range(E)}, x, sel, rw, H, I, bits)
    xt = torch.from_numpy(x.view(np.int16)).view(torch.bfloat16).to(DEV)
    for on in ("cpu", DEV):
        got = kernels.moe_prefill(torch.from_numpy(pool).to(DEV), {e: e for e in range(E)}, xt,
                                  torch.from_numpy(sel).to(on), torch.from_numpy(rw).to(DEV), n, H, I, bits)
        # the oracle's activation is rounded to bf16 as the kernels' is; one more rounding of the result
        err = np.linalg.norm(got.double().cpu().numpy() - ref) / np.linalg.norm(ref)
        assert err <= 2.0**-8, (on, err)


# x of 2 GiB: gate_up in its register form (scales staged in LDS up to 16 K groups, read as needed past them), against the
# halves of the tokens, whose x the LDS-DMA form takes: the same bits. 3 experts, one of them without a slot
@pytest.mark.parametrize("bits", [4, 3, 2])
@pytest.mark.parametrize("H,I", [(2048, 256), (4096, 128)])
def test_prefill_of_two_gib_of_tokens(bits, H, I):
    n, T = H * I, (1 << 30) // H
    rng = np.random.default_rng(H + bits)
    pool = torch.from_numpy(np.stack([O.quantize((rng.standard_normal(3 * n) * 0.05).astype(np.float32), bits, 128)
                                      for _ in range(2)])).to(DEV)
    gen = torch.Generator(device=DEV).manual_seed(H)
    x = torch.empty((T, H), dtype=torch.bfloat16, device=DEV).normal_(generator=gen)
    sel = torch.randint(0, 3, (T, 1), generator=gen, device=DEV)
    rw = torch.rand((T, 1), generator=gen, device=DEV)
    slots = {0: 1, 1: 0}
    got = kernels.moe_prefill(pool, slots, x, sel, rw, n, H, I, bits)
    for t in (slice(0, T // 2), slice(T // 2, T)):
        want = kernels.moe_prefill(pool, slots, x[t], sel[t], rw[t], n, H, I, bits)
        assert torch.equal(got[t].view(torch.int16), want.view(torch.int16))
    # and against the bf16 weights in float32 on some tokens: products of bf16 values, one rounding of the activation and
    # one of the result
    some = torch.randint(0, T, (64,), generator=gen, device=DEV)
    W = quant.dequant_rows(pool, torch.tensor([1, 0], device=DEV), n, bits, 128).float()
    ref = torch.zeros((64, H), device=DEV)
    for e in range(2):
        g, u, d = W[e, 0].view(I, H), W[e, 1].view(I, H), W[e, 2].view(H, I)
        xs = x[some].float()
        a = (torch.nn.functional.silu(xs @ g.t()) * (xs @ u.t())).to(torch.bfloat16).float()
        ref += (sel[some] == e) * rw[some] * (a @ d.t())
    assert ((got[some].float() - ref).norm() / ref.norm()).item() <= 2.0**-7
