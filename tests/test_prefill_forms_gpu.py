"""The streaming forms of the bf16 prefill (attention_prefill_wide.hip) at the edges of prefill_plan: 8 query tokens
per workgroup behind a long past, 16 and 32 for longer prompts.  Expected values come from the CPU oracle, or from
torch fp32 on the same inputs where the oracle takes minutes."""
import numpy as np
import pytest
import torch

from helpers import HKV, HQ, D, assert_bf16_close, from_dev, normal, read_cache, rng
from raftinfer_amd import ops
from test_attention_gpu import S, run_prefill
from test_fused_gpu import _prefill_case

pytestmark = pytest.mark.gpu


def shifted(t, elements=4):
    """A copy of t that starts `elements` past an allocation (8 bytes for the default of 4 bf16 values)."""
    flat = torch.empty(t.numel() + elements, device=t.device, dtype=t.dtype)[elements:]
    return flat.copy_(t.flatten()).view(t.shape)


def attend(T, past, layout, seed, edit=None, place=lambda t: t, edit_all=None):
    """Output, torch fp32 reference (non-finite values of V taken as 0) and whether the cache was written as expected,
    for random inputs; edit(k, v) or edit_all(q, k, v) changes the rows [past + T][4][256] (and q)
    before the call, place puts gate and output."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda *shape: torch.randn(*shape, device="cuda", generator=g).to(torch.bfloat16)
    n = past + T
    q, gate, k, v = rnd(T, HQ, D), rnd(T, HQ, D), rnd(n, HKV, D), rnd(n, HKV, D)
    if edit is not None:
        edit(k, v)
    if edit_all is not None:
        edit_all(q, k, v)
    rows = torch.stack([k, v])  # token-major
    full = rows.clone()
    rows[:, past:] = 0
    cache = (rows.transpose(1, 2) if layout == 1 else rows).contiguous()
    gate, out = place(gate), place(torch.empty(T, HQ, D, device="cuda", dtype=torch.bfloat16))
    ops.qwen35_causal_attention(q, k[past:].contiguous(), v[past:].contiguous(), gate, out, cache, None,
                                S(T, HQ, HKV, D, n, past), 3, ops.Qwen35AttentionLaunchPolicy(1, 1, layout))
    torch.cuda.synchronize()
    qf = q.float().permute(1, 0, 2)
    kf, vf = (x.float().repeat_interleave(HQ // HKV, dim=1).permute(1, 0, 2).contiguous() for x in (k, v))
    vf = torch.where(torch.isfinite(vf), vf, torch.zeros_like(vf))
    s = torch.matmul(qf, kf.transpose(1, 2).contiguous()) / 16.0
    hidden = torch.arange(n, device="cuda")[None] > past + torch.arange(T, device="cuda")[:, None]
    s = s.masked_fill(hidden, float("-inf"))
    ref = torch.matmul(torch.softmax(s, dim=-1), vf).permute(1, 0, 2) * torch.sigmoid(gate.float())
    written = cache if layout == 0 else cache.transpose(1, 2)
    return out, ref, torch.equal(written, full)


# Both sides of every line of prefill_plan.  8 tokens per workgroup: a single ragged query tile, one key tile more or less
# than a round of four, the first contexts that take the form; 16: its first prompt with and without a past, its last
# (2176 keys), query and key tiles of every length, behind a past from 1344 and 1440 keys; 32 (from 2177 keys): prompts
# that end in every part of a query tile and of a key tile, an odd and an even number of key tiles.
@pytest.mark.parametrize("T,past", [(2, 1022), (7, 1050), (33, 1000), (511, 513), (512, 512), (513, 513), (577, 1055),
                                    (1025, 0), (1039, 0), (1040, 65), (1072, 31), (2049, 0), (2080, 0), (2081, 40),
                                    (2113, 7), (2, 1023), (512, 513), (513, 830), (513, 831), (577, 863), (833, 510),
                                    (833, 607), (1024, 416), (2176, 0), (2049, 128), (2177, 0), (2208, 0), (2209, 40),
                                    (2241, 7)])
@pytest.mark.parametrize("layout", [0, 1])
def test_streaming_forms_against_torch(gpu, T, past, layout):
    out, ref, same = attend(T, past, layout, seed=T + past)
    assert same, "appended rows"
    assert_bf16_close(from_dev(out), from_dev(ref), what=f"prefill T={T} past={past} layout={layout}")


@pytest.mark.parametrize("T,past", [(40, 1000), (700, 600), (540, 920)])
def test_streaming_forms_against_oracle(gpu, T, past):
    out, expect, cache, keys, vals = run_prefill(3, 1, 1, T, HQ, HKV, D, past, seed=T)
    assert_bf16_close(out, expect, what=f"prefill T={T} past={past}")
    ck, cv = read_cache(cache, 1, past + T, past + T)
    assert np.array_equal(ck, keys) and np.array_equal(cv, vals)


def score_ramp(T, past, direction):
    """q [T][16][256] and k, v [past + T][4][256] whose scores run from -80 to +80 over the keys (or back): ascending,
    the reference max moves on every tile of every wave; descending, the first keys hold all the weight."""
    n = past + T
    ramp = (-80.0 + 160.0 * np.arange(n) / (n - 1)) * direction
    q = np.zeros((T, HQ, D), np.float32)
    q[:, :, 0] = 16.0
    k = np.zeros((n, HKV, D), np.float32)
    k[:, :, 0] = ramp[:, None]
    v = np.zeros((n, HKV, D), np.float32)
    for h in range(HKV):
        v[:, h] = 0.01 * (np.arange(n)[:, None] % 97 + np.arange(D)[None, :] + h)
    return q, k, v


@pytest.mark.parametrize("direction", [1, -1])
@pytest.mark.parametrize("T,past", [(64, 1100), (600, 520), (600, 900)])
def test_streaming_forms_rescale(gpu, direction, T, past):
    q, k, v = score_ramp(T, past, direction)
    out, expect, *_ = run_prefill(3, 1, 1, T, HQ, HKV, D, past,
                                  inputs=(q, normal(rng(5), T, HQ, D), k[past:], v[past:], k[:past], v[:past]))
    assert_bf16_close(out, expect, what=f"ramp {direction} T={T} past={past}")


@pytest.mark.parametrize("direction", [1, -1])
@pytest.mark.parametrize("layout", [0, 1])
def test_32_token_form_rescale(gpu, direction, layout):
    # (torch fp32 on the bf16 inputs: the oracle takes minutes here)
    T, past = 2200, 40
    ramp = torch.from_numpy(score_ramp(T, past, direction)[1]).cuda()

    def edit_all(q, k, v):
        q.zero_()
        q[:, :, 0] = 16.0
        k.copy_(ramp)

    out, ref, same = attend(T, past, layout, seed=9, edit_all=edit_all)
    assert same, "appended rows"
    assert_bf16_close(from_dev(out), from_dev(ref), what=f"ramp {direction} T={T} past={past} layout={layout}")


# A V row with an infinity or a NaN reaches exactly the tokens that see its key, as in a scalar sum: a masked key has
# probability 0, and 0 times such a value must not count.  Hit are a past row (if there is one), the first and the
# last new token, two neighbours inside a query tile and one in a later key tile of it, each in a dim of its own.
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("T,past,layout", [(600, 1020, 0), (600, 1020, 1), (1030, 0, 1), (1041, 0, 0), (1041, 30, 1),
                                           (2049, 0, 1), (2049, 0, 0), (2081, 40, 1), (2177, 0, 1), (2177, 0, 0),
                                           (2209, 40, 1)])
def test_streaming_forms_non_finite_values_reach_only_their_readers(gpu, T, past, layout, value):
    def readers(hits):  # first new token that sees each hit (dim, past + token)
        first = torch.full((D,), T, device="cuda")
        for d, row in hits:
            first[d] = max(0, row - past)
        return torch.arange(T, device="cuda")[:, None] >= first[None]  # [T][D]

    tokens = sorted({0, 8, 9, 17, 30, T - 1} & set(range(T)))
    hits = [(3 + 31 * i, past + t) for i, t in enumerate(tokens)] + ([(250, past - 1)] if past else [])

    def edit(k, v):
        for d, row in hits:
            v[row, 1, d] = value

    out, ref, same = attend(T, past, layout, seed=T + past, edit=edit)
    seen = torch.zeros(T, HQ, D, dtype=torch.bool, device="cuda")
    seen[:, 4:8] = readers(hits)[:, None]  # query heads of KV head 1
    got = out.float()
    assert torch.isnan(got[seen]).all() if value != value else (got[seen] == value).all()
    clean = torch.where(seen, torch.zeros_like(got), got)
    assert torch.isfinite(clean).all(), "a token that does not see the key"
    want = torch.where(seen, torch.zeros_like(ref), ref)
    assert_bf16_close(from_dev(clean), from_dev(want), what=f"prefill T={T} past={past} layout={layout}")


@pytest.mark.parametrize("T,past,rot,wdt,layout", [(17, 1011, 64, torch.bfloat16, 1), (100, 1000, 8, torch.float32, 0),
                                                   (520, 600, 256, torch.float32, 1), (1030, 0, 64, torch.bfloat16, 1),
                                                   (2050, 3, 192, torch.bfloat16, 0), (2079, 0, 256, torch.float32, 1),
                                                   (520, 960, 256, torch.float32, 1), (2178, 3, 192, torch.bfloat16, 0),
                                                   (2207, 0, 256, torch.float32, 1)])
def test_streaming_forms_fused_equal_producers_then_attention(gpu, T, past, rot, wdt, layout):
    c = _prefill_case(T, past, rot, wdt, layout, seed=T + past)
    assert torch.equal(c["cache1"], c["cache2"])
    assert torch.equal(c["out1"], c["out2"])


@pytest.mark.parametrize("T,past,rot,wdt,layout", [(521, 1000, 64, torch.bfloat16, 1), (1030, 0, 8, torch.float32, 0),
                                                   (2049, 3, 256, torch.float32, 1), (2080, 0, 24, torch.bfloat16, 0),
                                                   (2177, 3, 256, torch.float32, 1), (2208, 0, 24, torch.bfloat16, 0)])
def test_streaming_forms_fused_non_finite_values(gpu, T, past, rot, wdt, layout):
    # The same call with infinite values in a few tokens (the unfused one is compared with torch above).
    def edit(v):
        for t in (9, 300, 301, T - 1):
            v[t, 2, t % D] = np.inf

    c = _prefill_case(T, past, rot, wdt, layout, seed=T, edit_v=edit)
    out1, out2 = (c[x].view(T, HQ, D) for x in ("out1", "out2"))
    assert torch.isinf(out2[9:, 8:12, 9]).all() and torch.isfinite(out2[:9]).all()
    assert torch.isinf(out2).sum() == 4 * sum(T - t for t in (9, 300, 301, T - 1)) and not torch.isnan(out2).any()
    assert torch.equal(out1, out2) and torch.equal(c["cache1"], c["cache2"])


# Gate and output are accepted at 8-byte alignment, at sizes where each streaming form would take an aligned call.
@pytest.mark.parametrize("T,past,layout", [(10, 1020, 1), (600, 1020, 0), (1030, 0, 1), (2200, 0, 1)])
def test_gate_and_output_at_8_byte_alignment(gpu, T, past, layout):
    out, ref, same = attend(T, past, layout, seed=T, place=shifted)
    assert out.data_ptr() % 16 == 8
    assert same, "appended rows"
    assert_bf16_close(from_dev(out), from_dev(ref), what=f"prefill T={T} past={past} layout={layout}")


# ---- the f32 cache at the model shape (K, V and the probabilities at f32 precision; tiles of 16 keys, a round of 64)
def f32_cache(T, past, layout, seed, exact_bf16=False, edit=None, place=lambda t: t, query=None):
    g = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda *shape: torch.randn(*shape, device="cuda", generator=g)
    n = past + T
    q, gate = rnd(T, HQ, D).bfloat16(), rnd(T, HQ, D).bfloat16()
    if query is not None:
        q = query.bfloat16()
    rows = rnd(2, n, HKV, D)
    if exact_bf16:
        rows = rows.bfloat16().float()
    rows[:, past:] = rows[:, past:].bfloat16().float()
    if edit is not None:
        edit(rows)
    cache = rows.clone()
    cache[:, past:] = 0
    cache = (cache.transpose(1, 2) if layout == 1 else cache).contiguous()
    gate, out = place(gate), place(torch.empty(T, HQ, D, device="cuda", dtype=torch.bfloat16))
    ops.qwen35_causal_attention(q, rows[0, past:].bfloat16(), rows[1, past:].bfloat16(), gate, out, cache, None,
                                S(T, HQ, HKV, D, n, past), 3, ops.Qwen35AttentionLaunchPolicy(1, 0, layout))
    torch.cuda.synchronize()
    kf, vf = (x.double().repeat_interleave(HQ // HKV, dim=1).permute(1, 0, 2).contiguous() for x in rows)
    s = torch.matmul(q.double().permute(1, 0, 2), kf.transpose(1, 2).contiguous()) / 16.0
    hidden = torch.arange(n, device="cuda")[None] > past + torch.arange(T, device="cuda")[:, None]
    p = torch.softmax(s.masked_fill(hidden, float("-inf")), dim=-1)
    written = cache if layout == 0 else cache.transpose(1, 2)
    return out, p, vf, gate.double(), hidden, torch.equal(written, rows)


@pytest.mark.parametrize("T,past", [(2, 0), (9, 7), (16, 0), (17, 15), (65, 0), (64, 63), (100, 333), (512, 512)])
@pytest.mark.parametrize("layout,exact_bf16", [(0, True), (1, False), (0, False)])
def test_f32_cache_prefill(gpu, T, past, layout, exact_bf16):
    out, p, v, gate, _, same = f32_cache(T, past, layout, seed=T + past, exact_bf16=exact_bf16)
    assert same, "appended rows"
    want = (torch.matmul(p, v).permute(1, 0, 2) * torch.sigmoid(gate)).cpu().numpy()
    got = from_dev(out)
    # f32 sums of about 1e-6 of the largest product each, then one rounding to bf16 (2^-8 of the value at most)
    assert np.all(np.abs(got - want) <= 2.0 ** -8 * np.abs(want) * 1.001 + 2e-5)


@pytest.mark.parametrize("direction", [1, -1])
@pytest.mark.parametrize("layout,exact_bf16", [(0, True), (1, False), (1, True), (0, False)])
def test_f32_cache_prefill_rescale(gpu, direction, layout, exact_bf16):
    # The ramp over seven rounds of 64 keys: each wave's max moves by 12 to 24 log2 units from one of its tiles to its
    # next.  The values of the ramp that are not exact in bf16 take the products of the middle and low parts.
    T, past = 100, 333
    q, k, _ = (torch.from_numpy(x).cuda() for x in score_ramp(T, past, direction))

    def edit(rows):
        rows[0] = k.bfloat16().float() if exact_bf16 else k
        rows[0, past:] = rows[0, past:].bfloat16().float()

    out, p, v, gate, _, same = f32_cache(T, past, layout, seed=7, exact_bf16=exact_bf16, edit=edit, query=q)
    assert same, "appended rows"
    want = (torch.matmul(p, v).permute(1, 0, 2) * torch.sigmoid(gate)).cpu().numpy()
    got = from_dev(out)
    # scores to 80 carry 80 * 2^-23 each in f32 (3 of them: product, scale, maximum), which moves a weight by as much
    assert np.all(np.abs(got - want) <= (2.0 ** -8 * 1.001 + 3e-5) * np.abs(want) + 5e-5)


@pytest.mark.parametrize("T,past,layout,exact_bf16", [(40, 6000, 0, False), (9, 9001, 1, True), (1500, 70, 1, False)])
def test_f32_cache_prefill_many_rounds(gpu, T, past, layout, exact_bf16):
    out, p, v, gate, _, same = f32_cache(T, past, layout, seed=T, exact_bf16=exact_bf16)
    assert same, "appended rows"
    want = (torch.matmul(p, v).permute(1, 0, 2) * torch.sigmoid(gate)).cpu().numpy()
    assert np.all(np.abs(from_dev(out) - want) <= 2.0 ** -8 * np.abs(want) * 1.001 + 2e-5)


def test_f32_cache_prefill_gate_and_output_at_8_byte_alignment(gpu):
    out, p, v, gate, _, same = f32_cache(65, 70, 1, seed=8, place=shifted)
    assert same and out.data_ptr() % 16 == 8
    want = (torch.matmul(p, v).permute(1, 0, 2) * torch.sigmoid(gate)).cpu().numpy()
    assert np.all(np.abs(from_dev(out) - want) <= 2.0 ** -8 * np.abs(want) * 1.001 + 2e-5)


def test_f32_cache_prefill_keeps_bits_below_bf16(gpu):
    # Keys that differ only below bf16 decide the result: scores 1000 (1 + 2^-12 j) have softmax steps of 0.24 in j,
    # and in bf16 they would all be 1000.  V is the position, so the output is the mean position.
    T, n = 2, 40
    past = n - T
    rows = torch.zeros(2, n, HKV, D, device="cuda")
    j = torch.arange(past, device="cuda", dtype=torch.float32)
    rows[0, :past, :, 0] = (1000.0 * (1 + j * 2.0 ** -12))[:, None]
    rows[1, :past] = (j / past)[:, None, None]
    q = torch.zeros(T, HQ, D, device="cuda", dtype=torch.bfloat16)
    q[:, :, 0] = 16.0  # score = q.k / 16 = k[0]
    out = torch.empty(T, HQ, D, device="cuda", dtype=torch.bfloat16)
    zero = torch.zeros(T, HKV, D, device="cuda", dtype=torch.bfloat16)
    ops.qwen35_causal_attention(q, zero, zero, torch.zeros_like(q), out, rows, None, S(T, HQ, HKV, D, n, past), 3,
                                ops.Qwen35AttentionLaunchPolicy(1, 0, 0))
    torch.cuda.synchronize()
    p = torch.softmax(rows[0, :past, 0, 0].double(), 0)
    want = 0.5 * (p * rows[1, :past, 0, 0].double()).sum().item()  # the new keys' weight is e^-1000
    # bf16 rounding of the output; a score of 1000 carries 6e-5 in f32, which moves each weight by as much
    assert abs(out[0, 0, 0].item() - want) <= (2.0 ** -8 + 1e-3) * want


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
def test_f32_cache_prefill_infinite_values(gpu, value):
    # An infinite V row reaches exactly the tokens that see it, on past and new rows, as in a scalar sum.
    T, past = 20, 21
    rows_hit = [5, past + 7]

    def edit(rows):
        for r in rows_hit:
            rows[1, r, 1, 3] = value

    out, p, v, gate, hidden, _ = f32_cache(T, past, 0, seed=3, edit=edit)
    got = from_dev(out)
    finite = torch.where(torch.isfinite(v), v, torch.zeros_like(v))
    want = (torch.matmul(p, finite).permute(1, 0, 2) * torch.sigmoid(gate)).cpu().numpy()
    # every token sees row 5; column (head 4..7, dim 3) is infinite (NaN for NaN), all others as without it
    hit = np.zeros_like(want, bool)
    hit[:, 4:8, 3] = True
    assert np.all(np.abs(got - want)[~hit] <= 2.0 ** -8 * np.abs(want[~hit]) * 1.001 + 2e-5)
    assert np.isnan(got[hit]).all() if np.isnan(value) else (got[hit] == value).all()

    def edit_new(rows):
        rows[1, past + 7, 1, 3] = value

    out, p, v, gate, hidden, _ = f32_cache(T, past, 0, seed=3, edit=edit_new)
    got = from_dev(out)
    assert np.isfinite(got[:7]).all() and not np.isfinite(got[7:, 4:8, 3]).any()
    mask = np.ones_like(got, bool)
    mask[7:, 4:8, 3] = False
    assert np.isfinite(got[mask]).all()
