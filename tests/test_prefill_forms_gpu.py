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


def attend(T, past, layout, seed):
    """Output, torch fp32 reference and cache (as written, [2][4][ctx][256]) of random inputs."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda *shape: torch.randn(*shape, device="cuda", generator=g).to(torch.bfloat16)
    n = past + T
    q, gate, k, v = rnd(T, HQ, D), rnd(T, HQ, D), rnd(n, HKV, D), rnd(n, HKV, D)
    rows = torch.stack([k, v])  # token-major
    full = rows.clone()
    rows[:, past:] = 0
    cache = (rows.transpose(1, 2) if layout == 1 else rows).contiguous()
    out = torch.empty(T, HQ, D, device="cuda", dtype=torch.bfloat16)
    ops.qwen35_causal_attention(q, k[past:].contiguous(), v[past:].contiguous(), gate, out, cache, None,
                                S(T, HQ, HKV, D, n, past), 3, ops.Qwen35AttentionLaunchPolicy(1, 1, layout))
    torch.cuda.synchronize()
    qf = q.float().permute(1, 0, 2)
    kf, vf = (x.float().repeat_interleave(HQ // HKV, dim=1).permute(1, 0, 2).contiguous() for x in (k, v))
    s = torch.matmul(qf, kf.transpose(1, 2).contiguous()) / 16.0
    hidden = torch.arange(n, device="cuda")[None] > past + torch.arange(T, device="cuda")[:, None]
    s = s.masked_fill(hidden, float("-inf"))
    ref = torch.matmul(torch.softmax(s, dim=-1), vf).permute(1, 0, 2) * torch.sigmoid(gate.float())
    written = cache if layout == 0 else cache.transpose(1, 2)
    return out, ref, torch.equal(written, full)


# 8 tokens per workgroup: a single ragged query tile, one key tile more or less than a round of four, the first
# contexts that take the form; 16: its first prompt with and without a past; 32: prompts that end in every part of a
# query tile and of a key tile, an odd and an even number of key tiles.
@pytest.mark.parametrize("T,past", [(2, 1022), (7, 1050), (33, 1000), (511, 513), (512, 512), (513, 513), (577, 1055),
                                    (1025, 0), (1039, 0), (1040, 65), (1072, 31), (2049, 0), (2080, 0), (2081, 40),
                                    (2113, 7)])
@pytest.mark.parametrize("layout", [0, 1])
def test_streaming_forms_against_torch(gpu, T, past, layout):
    out, ref, same = attend(T, past, layout, seed=T + past)
    assert same, "appended rows"
    assert_bf16_close(from_dev(out), from_dev(ref), what=f"prefill T={T} past={past} layout={layout}")


@pytest.mark.parametrize("T,past", [(40, 1000), (700, 600)])
def test_streaming_forms_against_oracle(gpu, T, past):
    out, expect, cache, keys, vals = run_prefill(3, 1, 1, T, HQ, HKV, D, past, seed=T)
    assert_bf16_close(out, expect, what=f"prefill T={T} past={past}")
    ck, cv = read_cache(cache, 1, past + T, past + T)
    assert np.array_equal(ck, keys) and np.array_equal(cv, vals)


@pytest.mark.parametrize("direction", [1, -1])
@pytest.mark.parametrize("T,past", [(64, 1100), (600, 520)])
def test_streaming_forms_rescale(gpu, direction, T, past):
    # A -80 .. +80 score ramp: ascending, the reference max moves on every tile of every wave; descending, the first
    # keys hold all the weight.
    n = past + T
    ramp = (-80.0 + 160.0 * np.arange(n) / (n - 1)) * direction
    q = np.zeros((T, HQ, D), np.float32)
    q[:, :, 0] = 16.0
    k = np.zeros((n, HKV, D), np.float32)
    k[:, :, 0] = ramp[:, None]
    v = np.zeros((n, HKV, D), np.float32)
    for h in range(HKV):
        v[:, h] = 0.01 * (np.arange(n)[:, None] % 97 + np.arange(D)[None, :] + h)
    out, expect, *_ = run_prefill(3, 1, 1, T, HQ, HKV, D, past,
                                  inputs=(q, normal(rng(5), T, HQ, D), k[past:], v[past:], k[:past], v[:past]))
    assert_bf16_close(out, expect, what=f"ramp {direction} T={T} past={past}")


@pytest.mark.parametrize("T,past,rot,wdt,layout", [(17, 1011, 64, torch.bfloat16, 1), (100, 1000, 8, torch.float32, 0),
                                                   (520, 600, 256, torch.float32, 1), (1030, 0, 64, torch.bfloat16, 1),
                                                   (2050, 3, 192, torch.bfloat16, 0), (2079, 0, 256, torch.float32, 1)])
def test_streaming_forms_fused_equal_producers_then_attention(gpu, T, past, rot, wdt, layout):
    c = _prefill_case(T, past, rot, wdt, layout, seed=T + past)
    assert torch.equal(c["cache1"], c["cache2"])
    assert torch.equal(c["out1"], c["out2"])
