"""Parity at the benchmarked prefill sizes, on the kernels those sizes run.

A Qwen3-MoE-shaped layer (4096 tokens, 128 experts, Zipf(1.1) router skew)
and a mixed-width one (2048 tokens, 256 experts, 3-bit gate/up, 6-bit down,
sigmoid-gated shared expert) go through the grouped GEMM on the matrix cores;
each test first asserts that path (moe_layer_path). For every token the expert
ids, the f32 combine weights and the dispatch permutation / CSR offsets are
bit-exact against the oracle routing from the GPU's logits, and the logits are
within two storage ulps of the oracle's. The float output is checked against
the fp32-accumulated oracle on a sample of tokens chosen to cover the hottest
expert, the coldest used expert, experts whose last row tile is of each height,
tile boundaries and random tokens: a token's output depends only on its own
input row and routing, so the oracle runs on the sampled rows with their GPU
logits.

The literal bar, max |d| <= 2e-2 and mean |d| / mean |ref| <= 1e-3
with no rescaling, is asserted on layers whose weights are centred the way
mlx checkpoints are (bias about -scale * (2^bits - 1) / 2), so outputs are
O(1), on the one-token, batched matrix-core GEMV and grouped-GEMM paths."""
import ctypes as C

import numpy as np
import pytest

import oracle as orc
from moe_spec import (BF16, F16, LayerSpec, cfg_bits, cfg_gptoss, cfg_mixed, cfg_nemotron, cfg_qwen3,
                      check_close, gen_qproj,
                      load, store, to_numpy_f32, to_torch, zipf_router_bias, ZIPF_BETA)

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from ffai_amd import _lib  # noqa: E402
from ffai_amd._lib import check  # noqa: E402

# Row tiles of the grouped GEMM and the heights a last tile takes (the tall
# kernel: 256 rows)
GEMM_ROWS, GEMM_HEIGHTS = 96, (32, 64, 96)
TALL_ROWS, TALL_HEIGHTS = 256, (64, 128, 256)


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    _lib.load()
    yield
    torch.cuda.synchronize()


def _u32(t):
    return t.cpu().numpy().view(np.uint32)


def layer_paths(dev, T):
    p = _lib.LayerPaths()
    check(_lib.load().moe_layer_path(C.byref(dev.desc), T, C.byref(p)))
    return p.names()


def sample_tokens(idx, E, n_random, seed, rows=GEMM_ROWS, heights=GEMM_HEIGHTS):
    """Tokens covering the hottest and the coldest used expert, the first and
    last row of the last tile of up to 12 experts for each height that tile can
    take, the first and last row of every tile of the hottest expert, plus random
    tokens."""
    T, k = idx.shape
    counts = np.bincount(idx.ravel(), minlength=E)
    used = np.nonzero(counts)[0]
    hot, cold = int(np.argmax(counts)), int(used[np.argmin(counts[used])])
    rows_of = {e: np.nonzero((idx == e).any(axis=1))[0] for e in used}  # token order = plan order
    pick = set()
    for e in (hot, cold):
        r = rows_of[e]
        pick.update(r[[0, len(r) // 2, len(r) - 1]].tolist())
    by_height = {h: [] for h in heights}
    for e in used:
        last = (counts[e] - 1) % rows + 1
        by_height[next(h for h in heights if last <= h)].append(e)
    for es in by_height.values():
        for e in es[:12]:
            r = rows_of[e]
            pick.update((int(r[(len(r) - 1) // rows * rows]), int(r[-1])))
    r = rows_of[hot]
    for t0 in range(0, len(r), rows):
        pick.add(int(r[t0]))
        pick.add(int(r[min(t0 + rows, len(r)) - 1]))
    rng = np.random.default_rng(seed)
    pick.update(rng.choice(T, size=n_random, replace=False).tolist())
    return np.array(sorted(pick)), dict(hot=hot, cold=cold, hot_rows=int(counts[hot]),
                                        cold_rows=int(counts[cold]),
                                        heights={h: len(es) for h, es in by_height.items()})


def run_full(spec, T, expect, seed=0, n_random=48, tiles=(GEMM_ROWS, GEMM_HEIGHTS)):
    dev = spec.device()
    paths = layer_paths(dev, T)
    for key, val in expect.items():
        assert paths[key] == val, f"{spec.name} T={T}: {key} runs {paths[key]}, expected {val}"
    x = spec.x(T, seed)
    y, tr = dev.forward(to_torch(x), trace=True)
    torch.cuda.synchronize()
    logits_gpu = to_numpy_f32(tr["logits"])
    logits_cpu = spec.oracle_logits(x)
    assert np.all(np.abs(logits_gpu - logits_cpu) <= spec.logits_tolerance(logits_cpu)), \
        "router logits"
    # routing and plan for every token, from the GPU logits
    idx_ref, w_ref = orc.route(logits_gpu, spec.top_k, spec.gating, spec.norm_topk,
                               spec.expert_bias, spec.logit_scale, spec.routed_scale,
                               spec.expert_scale)
    assert np.array_equal(_u32(tr["topk_idx"]), idx_ref), "expert ids"
    assert np.array_equal(tr["topk_weight"].cpu().numpy().view(np.uint32), w_ref.view(np.uint32)), \
        "combine weights"
    _, off_ref, perm_ref, _ = orc.dispatch_plan(idx_ref, spec.n_experts)
    assert np.array_equal(_u32(tr["perm"]), perm_ref), "dispatch permutation"
    assert np.array_equal(_u32(tr["offsets"]), off_ref), "CSR offsets"
    # float output on the sampled tokens
    toks, info = sample_tokens(idx_ref, spec.n_experts, n_random, seed, *tiles)
    assert len(toks) >= 64, len(toks)
    y_ref, _, idx_s, _ = orc.moe_layer(spec, x[toks], given_logits=logits_gpu[toks])
    assert np.array_equal(idx_s, idx_ref[toks])
    got = to_numpy_f32(y)[toks]
    stats = check_close(got, load(y_ref, spec.act_dt), spec.act_dt, f"{spec.name} T={T}")
    print(f"{spec.name} T={T} paths={paths} sampled {len(toks)} tokens {info}: "
          f"max|d|/scale={stats[0]:.3e} mean_rel={stats[1]:.3e}")
    return info


def test_prefill_4096_zipf_full_size():
    """4096 tokens, 128 experts, top-8, Zipf(1.1) skew calibrated to
    a hottest-expert load of about 10x the median."""
    spec = cfg_qwen3(seed=5, router_bias=zipf_router_bias(128, 1.1, beta=ZIPF_BETA))
    info = run_full(spec, 4096, dict(gate_up="gemm", down="gemm"))
    assert all(info["heights"].values()), info


def test_mixed_2048_shared_full_size():
    """2048 tokens, 256 experts, 3-bit gate/up and 6-bit down, and
    the sigmoid-gated shared expert on its side stream."""
    info = run_full(cfg_mixed(), 2048, dict(gate_up="gemm", down="gemm", shared_gate_up="gemm",
                                            shared_down="gemm"))
    assert info["hot_rows"] > 0


def test_gptoss_256_gemm_path():
    """GPT-OSS-20B shape (hidden = intermediate = 2880, 32 experts, top-4, the
    biased router, per-expert output biases and the clamped SwiGLU) at 256
    tokens: 32 rows per expert take the grouped GEMM, and the router
    projection writes the GEMMs' f16 operand copy from its LDS chunks (2880 =
    11.25 chunks of 256, so the last chunk's pieces past the row end are
    dropped)."""
    info = run_full(cfg_gptoss(seed=7, expert_bias=True), 256, dict(gate_up="gemm", down="gemm"))
    assert info["hot_rows"] > 0


def _many_rows(kind):
    if kind == "gptoss":  # per-expert output biases, clamped SwiGLU
        return cfg_gptoss(seed=8, n_experts=8, expert_bias=True), 2048
    if kind == "relu2":   # one up projection, whose activation is the down GEMM's operand
        return cfg_nemotron(seed=9, n_experts=8, hidden=2048, inter=5888, top_k=4), 2048
    gu, dn, gs, sb, dt = kind
    return cfg_bits(gu, dn, gs, sb, dt, seed=10, hidden=2048, inter=2880, n_experts=8, top_k=2), 4096


@pytest.mark.parametrize("kind", ["gptoss", "relu2", (4, 4, 64, F16, BF16), (3, 6, 32, BF16, BF16),
                                  (8, 8, 64, F16, F16), (6, 4, 64, BF16, BF16)], ids=str)
def test_many_rows_per_expert(kind):
    """1024 rows per expert on average and more than 700 blocks of 256 rows x
    256 weight rows: the grouped GEMM's 256-row tiles for the gate/up pair (or
    the single up projection) and the down projection."""
    spec, T = _many_rows(kind)
    run_full(spec, T, dict(gate_up="gemm", down="gemm"), tiles=(TALL_ROWS, TALL_HEIGHTS))


# ------------------------------------------------- the literal float bar --

def cfg_centred(seed, E, H, I, k, bits_gu=4, bits_d=4, act_dt=BF16, sb_dt=BF16, shared=False):
    """A layer whose dequantised weights are centred on zero (bias about
    -scale * (2^bits - 1) / 2, as mlx's affine quantiser produces) with scales
    sized so that the layer's outputs are O(1)."""
    rng = np.random.default_rng(seed)

    def proj(E_, n, kk, bits):
        f = 15.0 / (2 ** bits - 1)
        lo, hi = 0.8 * f / np.sqrt(kk) * 0.25, 1.2 * f / np.sqrt(kk) * 0.25
        q = gen_qproj(rng, E_, n, kk, bits, 64, sb_dt, s_range=(lo, hi))
        s = load(q.scales, sb_dt)
        b = -s * (2 ** bits - 1) / 2 + rng.normal(0, 0.05, size=s.shape) * s
        return orc.QProj(q.weight, q.scales, store(b, sb_dt), bits, 64, sb_dt)

    sh = None
    sgw = None
    if shared:
        sh = (proj(1, I, H, bits_gu), proj(1, I, H, bits_gu), proj(1, H, I, bits_d))
        sgw = store(rng.normal(0, 1 / np.sqrt(H), size=(1, H)), act_dt)
    return LayerSpec(H, E, k, I, act_dt,
                     router_weight=store(rng.normal(0, 1 / np.sqrt(H), size=(E, H)), act_dt),
                     router_dt=act_dt, gate=proj(E, I, H, bits_gu), up=proj(E, I, H, bits_gu),
                     down=proj(E, H, I, bits_d), shared=sh, shared_gate_weight=sgw,
                     name=f"centred{bits_gu}/{bits_d}")


def literal_bar(got, ref, label):
    d = np.abs(np.asarray(got, np.float64) - np.asarray(ref, np.float64))
    max_abs = float(d.max())
    mean_rel = float(d.mean() / np.abs(ref).mean())
    print(f"{label}: max|d|={max_abs:.3e} mean_rel={mean_rel:.3e} rms(ref)="
          f"{float(np.sqrt(np.mean(np.square(ref)))):.3f} max|ref|={float(np.abs(ref).max()):.3f}")
    assert max_abs <= 2e-2, f"{label}: max |d| = {max_abs:.3e} > 2e-2"
    assert mean_rel <= 1e-3, f"{label}: mean relative error {mean_rel:.3e} > 1e-3"


@pytest.mark.parametrize("T,path,E,k,bits", [
    (1, "decode1", 128, 8, (4, 4)),      # one token, fused kernels
    (1, "decode1", 256, 8, (3, 6)),
    (64, "gemv_mma", 128, 8, (4, 4)),    # 4 rows per used expert on the matrix cores
    (64, "gemv_mma", 256, 8, (3, 6)),
    (1024, "gemm", 32, 4, (4, 4)),       # grouped GEMM, 128 rows per expert
    (1024, "gemm", 32, 4, (3, 6)),
    (256, "gemm", 16, 4, (4, 4)),        # 64 rows per expert: 64- and 96-row tiles
    (320, "gemm", 16, 4, (3, 6)),        # 80 rows per expert
])
def test_literal_tolerance_centred(T, path, E, k, bits):
    spec = cfg_centred(seed=T + E, E=E, H=2048, I=768, k=k, bits_gu=bits[0], bits_d=bits[1])
    dev = spec.device()
    assert layer_paths(dev, T)["gate_up"] == path
    x = spec.x(T, seed=3)
    y, tr = dev.forward(to_torch(x), trace=True)
    torch.cuda.synchronize()
    logits = to_numpy_f32(tr["logits"])
    n = min(T, 96)
    y_ref, _, idx_ref, _ = orc.moe_layer(spec, x[:n], given_logits=logits[:n])
    assert np.array_equal(_u32(tr["topk_idx"])[:n], idx_ref)
    literal_bar(to_numpy_f32(y)[:n], load(y_ref, spec.act_dt), f"{spec.name} T={T} {path}")
