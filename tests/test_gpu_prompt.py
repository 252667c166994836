"""The wide products of a resident prompt (kernels.prompt_i8 and prompt_fp8) at the edges of their tiles, against the
32-row products (grouped_i8, themselves pinned on the oracle) on the same planes, and their decoding against the
oracle's. resident_prefill's own oracle tests with many rows per expert run through them too."""
import numpy as np
import pytest
import torch

from drama3 import kernels, offload
from oracle import numerics
from oracle import reference as ref
from tests.test_gpu_ref import DEV, _bank, dev, fields_on, zipf_topk

pytestmark = pytest.mark.gpu

# rows per expert: none, one, around one 16-row tile, around a pass's 96 rows, two and three passes, an odd middle
COUNTS = [0, 1, 15, 16, 17, 95, 96, 97, 193, 240, 50]


@pytest.mark.parametrize("E, P", [(1, 1), (7, 1023), (128, 1025), (256, 30011), (1024, 70000), (100, 131072 + 5)])
def test_prompt_groups(E, P):
    """The grouping over many workgroups, from one pair to more than 64 blocks of 1024 of them, some ids outside the
    experts: every pair once, the experts in ascending order, inverse the pairs' places (-1 and after every group for
    an id outside), and passes that cover each expert's places in runs of at most 96, those of most tiles first."""
    rng = np.random.default_rng(E)
    ids = rng.integers(0, E, P)
    ids[rng.random(P) < 0.3] = E // 2
    bad = rng.random(P) < 0.01
    ids[bad] = rng.choice([-1, E, E + 5, -2 ** 40, 2 ** 40], size=int(bad.sum()))
    order, inverse, passes = (t.cpu().numpy() for t in kernels.prompt_groups(dev(ids.astype(np.int64)).view(-1, 1), E))
    assert np.array_equal(np.sort(order), np.arange(P))
    valid = (ids >= 0) & (ids < E)
    n = int(valid.sum())
    assert np.array_equal(ids[order[:n]], np.sort(ids[valid])) and not valid[order[n:]].any()
    assert np.array_equal(inverse[order[:n]], np.arange(n)) and np.all(inverse[~valid] == -1)
    listed = passes[4:4 + 4 * passes[0]].reshape(-1, 4)
    tiles = (listed[:, 2] + 15) // 16
    assert np.all(listed[:, 2] >= 1) and np.all(tiles <= 6)
    counts = np.bincount(ids[valid], minlength=E)
    first = np.cumsum(counts) - counts
    for e in np.unique(ids[valid]):
        own = listed[listed[:, 0] == e]
        own = own[np.argsort(own[:, 1])]
        assert own[0, 1] == first[e] and np.array_equal(own[1:, 1], own[:-1, 1] + own[:-1, 2])
        assert own[:, 2].sum() == counts[e] and len(set(((own[:-1, 2] + 15) // 16).tolist())) <= 1
    assert set(listed[:, 0].tolist()) == set(np.unique(ids[valid]).tolist())


@pytest.mark.parametrize("K, N", [(256, 512), (2048, 256), (768, 1024)])
@pytest.mark.parametrize("kind", ["int8", "w4", "w6"])
def test_prompt_products_match_the_32_row_products(kind, K, N):
    """Both read the same int8 planes and add the same exact int32 sums A0, A1, A2 in float32, A0 + (A1 + A2 / 254) /
    254, each step rounded once: bit for bit the same. SwiGLU: SiLU(gate) * up of the same numbers, with a float32 exp
    and divide (2^-20)."""
    rng = np.random.default_rng(len(kind) + K)
    E, T = len(COUNTS), sum(COUNTS)
    fields = fields_on(_bank(kind, rng, E, N, K))
    cb = dev(ref.default_codebook()) if kind == "w4" else None
    idx = dev(rng.permutation(np.repeat(np.arange(E), COUNTS)).astype(np.int64)).view(T, 1)
    x = dev(rng.standard_normal((T, K)).astype(np.float32)).to(torch.bfloat16)
    order, inverse, passes, planes, scales = kernels.prompt_prep_i8(idx, E, x, True)
    listed = passes[4:4 + 4 * int(passes[0])].view(-1, 4).cpu().numpy()
    assert listed[:, 2].sum() == T and listed[:, 2].min() >= 1 and listed[:, 2].max() <= 96
    order2, inverse2, groups, work, planes2, scales2 = kernels.expert_groups_prep_i8(idx, E, x, True)
    assert torch.equal(planes, planes2) and torch.equal(scales, scales2)
    got = kernels.prompt_i8(kind, planes, scales, T, K, passes, E, fields, cb, N, order, 1)
    want = kernels.grouped_i8(kind, planes, scales, T, K, groups, work, fields, fields, cb, N, order=order2, k=1)
    got, want = got[inverse.long()].double(), want[inverse2.long()].double()  # by token
    assert torch.equal(got, want)
    hidden = kernels.prompt_i8(kind, planes, scales, T, K, passes, E, fields, cb, N, order, 1, swiglu=True)
    gate, up = got[:, :N // 2], got[:, N // 2:]
    want = gate / (1 + torch.exp(-gate)) * up
    assert torch.all((hidden[inverse.long()].double() - want).abs() <= 2.0 ** -20 * (want.abs() + gate.abs() * 1e-6))


def test_planes_meet_by_two_divisions():
    """The int8 products' float32 epilogue, scale * (S * (A0 + (A1 + A2 / 254) / 254)) with every step rounded once, bit
    for bit numpy's on the exact sums, in the wide and in the 32-row products."""
    rng = np.random.default_rng(254)
    E, N, K, T = 2, 512, 2048, 200
    host = _bank("int8", rng, E, N, K)
    idx = dev(np.arange(T, dtype=np.int64) % E).view(T, 1)
    x = dev(rng.standard_normal((T, K)).astype(np.float32)).to(torch.bfloat16)
    order, inverse, passes, planes, scales = kernels.prompt_prep_i8(idx, E, x, True)
    order2, inverse2, groups, work, planes2, scales2 = kernels.expert_groups_prep_i8(idx, E, x, True)
    fields = fields_on(host)
    wide = kernels.prompt_i8("int8", planes, scales, T, K, passes, E, fields, None, N, order, 1)
    narrow = kernels.grouped_i8("int8", planes2, scales2, T, K, groups, work, fields, fields, None, N, order=order2, k=1)
    a = planes.view(3, T, K).double().cpu()
    sx = scales.cpu().numpy()[:, None]
    for e in range(E):
        w = torch.from_numpy(host["_qdata"][e * N:(e + 1) * N]).double()
        a0, a1, a2 = ((p[e::E] @ w.T).numpy().astype(np.float32) for p in a)  # under 2^25 in float64: exact
        ratio = np.float32(254)
        want = (host["scale"].reshape(-1)[e * N:(e + 1) * N].astype(np.float32)
                * (sx[e::E] * (a0 + (a1 + a2 / ratio) / ratio)))
        assert np.array_equal(wide[inverse.long()].cpu().numpy()[e::E], want)
        assert np.array_equal(narrow[inverse2.long()].cpu().numpy()[e::E], want)


@pytest.mark.parametrize("E, k, H, I", [(12, 4, 2048, 512), (5, 2, 768, 1024), (3, 1, 256, 256)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kind", ["int8", "fp8", "w4", "w6"])
def test_prompt_rows_do_not_depend_on_how_many_run(kind, dtype, E, k, H, I):
    """A row's result through the wide products, bit for bit the same rows' in prompts short enough for the 32-row ones."""
    rng = np.random.default_rng(len(kind) + E)
    T = 2077 // k + 1
    banks = [fields_on(b) for b in (_bank(kind, rng, E, 2 * I, H), _bank(kind, rng, E, H, I))]
    cb = dev(ref.default_codebook()) if kind == "w4" else None
    idx = dev(zipf_topk(rng, T, E, k).astype(np.int64))
    w = dev(rng.dirichlet(np.ones(k), T).astype(np.float32))
    x = dev(rng.standard_normal((T, H)).astype(np.float32)).to(dtype)
    run = lambda s: offload.resident_prefill(x[s], idx[s], w[s], banks, (2 * I, H), kind, (cb, cb), E)  # noqa: E731
    fits = lambda n: kernels.prompt_wide_fits(kind, banks, (2 * I, H), n * k, E, H)  # noqa: E731
    assert fits(T) and not fits(200)
    assert torch.equal(run(slice(T)), torch.cat([run(slice(t, t + 200)) for t in range(0, T, 200)]))


@pytest.mark.parametrize("kind", ["w4", "w6"])
def test_prompt_products_decode_exactly(kind):
    """One-hot rows make each output one decoded weight times its channel scale, a single product: bit for bit the
    oracle's, for every scale byte but NaN's."""
    rng = np.random.default_rng(len(kind))
    E, N, K = 2, 256, 256
    host = _bank(kind, rng, E, N, K)
    finite = np.array([b for b in range(256) if b & 0x7F != 0x7F], np.uint8)
    host["scale"] = rng.choice(finite, size=host["scale"].shape)
    cb = ref.default_codebook()
    fields = fields_on(host)
    idx = dev(np.repeat(np.arange(E), K).astype(np.int64)).view(-1, 1)
    x = torch.eye(K, device=DEV).repeat(E, 1)
    order, inverse, passes, planes, scales = kernels.prompt_prep_i8(idx, E, x, False)
    out = kernels.prompt_i8(kind, planes, scales, E * K, K, passes, E, fields, dev(cb) if kind == "w4" else None, N,
                            order, 1)[inverse.long()].cpu().numpy()
    w = ref.decode_codes_ref(host["_qdata"], host["scale"], int(kind[1]), cb).astype(np.float32)
    w = w * host["s_channel"].reshape(-1, 1).astype(np.float32)
    for e in range(E):
        assert np.array_equal(out[e * K:(e + 1) * K], w[e * N:(e + 1) * N].T)


@pytest.mark.parametrize("planes", [1, 3])
@pytest.mark.parametrize("K, N", [(256, 512), (2048, 256), (768, 1024)])
def test_prompt_fp8_products_match_the_32_row_products(K, N, planes):
    """Over bf16 rows and over float32 rows as three planes: float32 sums of the same exact products in the same order, bit
    for bit."""
    rng = np.random.default_rng(K + planes)
    E, T = len(COUNTS), sum(COUNTS)
    host = _bank("fp8", rng, E, N, K)
    fields = fields_on(host)
    idx = dev(rng.permutation(np.repeat(np.arange(E), COUNTS)).astype(np.int64)).view(T, 1)
    x = dev(rng.standard_normal((T, K)).astype(np.float32))
    x = x.to(torch.bfloat16) if planes == 1 else x
    split = x.view(1, -1) if planes == 1 else kernels.prep_planes(x, False)
    order, inverse, passes = kernels.prompt_groups(idx, E)
    order2, inverse2, groups, work = kernels.expert_groups(idx, E, plan=True)
    got = kernels.prompt_fp8(split, T, K, passes, E, fields, N, order, 1)[inverse.long()].double()
    want = kernels.grouped_fp8_planes(split, T, K, groups, work, fields, fields, N, order=order2, k=1)
    want = want[inverse2.long()].double()
    assert torch.equal(got, want)
    hidden = kernels.prompt_fp8(split, T, K, passes, E, fields, N, order, 1, swiglu=True)[inverse.long()].double()
    gate, up = got[:, :N // 2], got[:, N // 2:]
    want = gate / (1 + torch.exp(-gate)) * up
    assert torch.all((hidden - want).abs() <= 2.0 ** -20 * (want.abs() + gate.abs() * 1e-6))


def test_prompt_fp8_products_decode_exactly():
    """One-hot rows make each output one e4m3 code times its block scale, bit for bit the oracle's."""
    rng = np.random.default_rng(8)
    E, N, K = 2, 256, 256
    host = _bank("fp8", rng, E, N, K)
    idx = dev(np.repeat(np.arange(E), K).astype(np.int64)).view(-1, 1)
    x = torch.eye(K, device=DEV, dtype=torch.bfloat16).repeat(E, 1)
    order, inverse, passes = kernels.prompt_groups(idx, E)
    out = kernels.prompt_fp8(x.view(1, -1), E * K, K, passes, E, fields_on(host), N, order, 1)[inverse.long()]
    w = ref.fp8_rows(host["weight"], host["scale"]).astype(np.float32)
    for e in range(E):
        assert np.array_equal(out[e * K:(e + 1) * K].cpu().numpy(), w[e * N:(e + 1) * N].T)


@pytest.mark.parametrize("kind", ["int8", "fp8", "w4", "w6"])
def test_prompt_path_equals_the_32_row_path_and_replays(kind, monkeypatch):
    """resident_prefill through the wide products and through the 32-row ones: the same bits; captured in a graph, every
    replay equals the eager result bit for bit, with other work in between."""
    rng = np.random.default_rng(30 + len(kind))
    E, T, k, H, I = 12, 555, 4, 2048, 512
    banks = [fields_on(b) for b in (_bank(kind, rng, E, 2 * I, H), _bank(kind, rng, E, H, I))]
    cb = dev(ref.default_codebook()) if kind == "w4" else None
    idx = dev(zipf_topk(rng, T, E, k).astype(np.int64))
    w = dev(numerics.bf16_round(rng.dirichlet(np.ones(k), T).astype(np.float32))).to(torch.bfloat16)
    x = dev(rng.standard_normal((T, H)).astype(np.float32)).to(torch.bfloat16)
    run = lambda: offload.resident_prefill(x, idx, w, banks, (2 * I, H), kind, (cb, cb), E)  # noqa: E731
    assert kernels.prompt_wide_fits(kind, banks, (2 * I, H), T * k, E, H)
    wide = run()
    monkeypatch.setattr(kernels, "PROMPT_WIDE_ROWS", 10 ** 9)
    narrow = run()
    monkeypatch.undo()
    assert torch.equal(wide.view(torch.int16), narrow.view(torch.int16))
    stream = torch.cuda.Stream(DEV)
    stream.wait_stream(torch.cuda.current_stream(DEV))
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        with torch.cuda.graph(g, stream=stream):
            out = run()
    torch.cuda.current_stream(DEV).wait_stream(stream)
    for _ in range(3):
        x.copy_(torch.randn(x.shape, device=DEV).to(torch.bfloat16))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), run().view(torch.int16))


def test_prompt_fp8_rows_at_any_storage_offset():
    """Contiguous bf16 rows that start one element into their storage (bf16 rows are FP8's plane as they are): the same
    result as the aligned rows, bit for bit, from as many rows as the wide products take."""
    rng = np.random.default_rng(40)
    E, T, k, H, I = 4, 1031, 2, 256, 256
    banks = [fields_on(b) for b in (_bank("fp8", rng, E, 2 * I, H), _bank("fp8", rng, E, H, I))]
    idx = dev(zipf_topk(rng, T, E, k).astype(np.int64))
    w = dev(rng.dirichlet(np.ones(k), T).astype(np.float32))
    x = dev(rng.standard_normal((T, H)).astype(np.float32)).to(torch.bfloat16)
    offset = torch.empty(T * H + 1, dtype=torch.bfloat16, device=DEV)[1:].view(T, H).copy_(x)
    assert offset.is_contiguous() and offset.data_ptr() % 16 == 2
    assert kernels.prompt_wide_fits("fp8", banks, (2 * I, H), T * k, E, H)
    got, want = (offload.resident_prefill(v, idx, w, banks, (2 * I, H), "fp8", (None, None), E) for v in (offset, x))
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
