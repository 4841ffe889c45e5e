"""Batched-prefill attention (forward_batch's per-token attention, mod.rs:1101-1140
over ops.rs:353-406) through hh_attention_prefill, against a float64 numpy
restatement of causal softmax attention:

  * mode 0, the split/merge kernels the batched prefill runs by default: within
    1e-5 of float64, and each token's row equal bit for bit to the decode
    operator hh_attention at seq_len pos0 + t + 1 (the prefill restates the
    decode order);
  * mode 1, the fp32-MFMA flash form (HH_PREFILL_ATTN=mfma): within 1e-5 of
    float64 (its sums are regrouped, so this is its parity bar).

Geometries cover head_dim 128 and 256, query groups 1, 3, 4, 6 and 8 (so the
MFMA kernel's workgroups of 4 tiles and of 1 tile; 2 tiles are tested below), partial 16-token tiles, a
prompt that starts past position 0 and one long enough for many chunks.  A
model-level check runs a 9B-shaped slice and an 8B-shaped slice through the
batched prefill both ways."""
import os

import numpy as np
import pytest

from hearth_amd.lib import CONFIGS

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _ref(q, k, v, pos0):
    n, nh, hd = q.shape
    nkv = k.shape[0]
    G = nh // nkv
    out = np.zeros((n, nh, hd))
    for t in range(n):
        L = pos0 + t + 1
        for h in range(nh):
            kk = k[h // G, :L].astype(np.float64)
            s = kk @ q[t, h].astype(np.float64) / np.sqrt(hd)
            p = np.exp(s - s.max())
            out[t, h] = (p / p.sum()) @ v[h // G, :L].astype(np.float64)
    return out


@pytest.mark.parametrize("nh,nkv,hd,pos0,n", [(32, 8, 128, 0, 300), (16, 4, 256, 37, 70), (16, 2, 128, 5, 50),
                                              (8, 8, 128, 0, 45), (24, 4, 256, 0, 33), (6, 2, 128, 100, 29)])
def test_prefill_attention_modes_vs_float64(ctx, nh, nkv, hd, pos0, n):
    rng = np.random.default_rng(nh * 1000 + hd + pos0 + n)
    ms = pos0 + n + 24
    q = rng.standard_normal((n, nh, hd)).astype(np.float32)
    k = rng.standard_normal((nkv, ms, hd)).astype(np.float32)
    v = rng.standard_normal((nkv, ms, hd)).astype(np.float32)
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()
    dq, dk, dv = dev(q), dev(k), dev(v)
    want = _ref(q, k, v, pos0)
    print(f"prefill attention {nh}/{nkv} x {hd}, pos0 {pos0}, {n} tokens", flush=True)
    got = {}
    for mode in (0, 1):
        out = torch.full((n * nh * hd,), float("nan"), dtype=torch.float32, device="cuda")
        ctx.attention_prefill(dq, dk, dv, nh, nkv, hd, ms, pos0, n, mode, out)
        ctx.sync()
        got[mode] = out.cpu().numpy().reshape(n, nh, hd)
        err = float(np.abs(got[mode] - want).max() / np.abs(want).max())
        print(f"  mode {mode}: max rel err vs float64 {err:.2e}", flush=True)
        assert np.isfinite(got[mode]).all() and err < 1e-5, (mode, err)
    # the default path is the decode operator's order, token by token
    for t in sorted({0, n // 2, n - 1}):
        one = torch.zeros(nh * hd, dtype=torch.float32, device="cuda")
        ctx.attention(dev(q[t]), dk, dv, nh, nkv, hd, ms, pos0 + t + 1, one)
        ctx.sync()
        assert np.array_equal(one.cpu().numpy(), got[0][t].reshape(-1)), t


@pytest.mark.parametrize("nh,nkv,hd,pos0,n", [
    (5, 1, 128, 0, 1), (7, 1, 256, 3, 17), (16, 8, 128, 15, 16),      # group sizes 5, 7, 2; one token, one tile
    (8, 8, 128, 2040, 41), (24, 4, 256, 2031, 49),                    # narrow to wide chunks inside the prompt
    (32, 8, 128, 63, 1100), (16, 4, 256, 0, 900)])                    # 16 to 64 tokens per workgroup
def test_prefill_split_equals_decode_at_edges(ctx, nh, nkv, hd, pos0, n):
    """The split pass on the matrix instructions restates the decode split bit for bit: the
    rows at tile, chunk and width edges equal hh_attention's, with the cache's rows past
    the prompt not numbers."""
    rng = np.random.default_rng(nh * 100 + hd + pos0 + n)
    ms = pos0 + n + 70
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()
    q = rng.standard_normal((n, nh, hd)).astype(np.float32)
    k = rng.standard_normal((nkv, ms, hd)).astype(np.float32) * 2
    v = rng.standard_normal((nkv, ms, hd)).astype(np.float32)
    k[:, pos0 + n:] = np.nan
    v[:, pos0 + n:] = np.nan
    dk, dv = dev(k), dev(v)
    out = torch.full((n * nh * hd + 64,), 7.0, dtype=torch.float32, device="cuda")
    print(f"prefill split {nh}/{nkv} x {hd}, pos0 {pos0}, {n} tokens", flush=True)
    ctx.attention_prefill(dev(q), dk, dv, nh, nkv, hd, ms, pos0, n, 0, out)
    ctx.sync()
    got = out.cpu().numpy()
    assert (got[n * nh * hd:] == 7.0).all()
    got = got[:n * nh * hd].reshape(n, -1)
    edges = {0, 1, 15, 16, 17, 31, 32, 63, 64, n // 2, n - 2, n - 1}
    edges |= {p - pos0 + d for p in (64, 128, 512, 1024, 2048) for d in (-2, -1, 0, 1)}   # chunks, the wide rule
    one = torch.zeros(nh * hd, dtype=torch.float32, device="cuda")
    for t in sorted(e for e in edges if 0 <= e < n):
        ctx.attention(dev(q[t]), dk, dv, nh, nkv, hd, ms, pos0 + t + 1, one)
        ctx.sync()
        assert np.array_equal(one.cpu().numpy(), got[t]), t


@pytest.mark.parametrize("nh,nkv,hd,pos0,n", [(16, 8, 128, 7, 49), (8, 8, 128, 0, 65), (2, 2, 256, 90, 63),
                                              (8, 4, 256, 31, 17), (9, 3, 128, 12, 33)])
def test_prefill_mfma_tiles_of_a_workgroup(ctx, nh, nkv, hd, pos0, n):
    """The matrix form with several 16-token tiles per workgroup (1 and 2 query heads per
    kv head) and one (3): a tile's rows equal, bit for bit, those of a call on that tile
    alone."""
    rng = np.random.default_rng(nh * 10 + hd + pos0 + n)
    ms = pos0 + n + 5
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()
    q = rng.standard_normal((n, nh, hd)).astype(np.float32)
    dk = dev(rng.standard_normal((nkv, ms, hd)).astype(np.float32) * 2)
    dv = dev(rng.standard_normal((nkv, ms, hd)).astype(np.float32))
    out = torch.full((n * nh * hd + 64,), 7.0, dtype=torch.float32, device="cuda")
    print(f"prefill mfma tiles {nh}/{nkv} x {hd}, pos0 {pos0}, {n} tokens", flush=True)
    ctx.attention_prefill(dev(q), dk, dv, nh, nkv, hd, ms, pos0, n, 1, out)
    ctx.sync()
    got = out.cpu().numpy()
    assert (got[n * nh * hd:] == 7.0).all()
    got = got[:n * nh * hd].reshape(n, -1)
    for t in range(0, n, 16):
        m = min(16, n - t)
        one = torch.zeros(m * nh * hd, dtype=torch.float32, device="cuda")
        ctx.attention_prefill(dev(q[t:t + m]), dk, dv, nh, nkv, hd, ms, pos0 + t, m, 1, one)
        ctx.sync()
        assert np.array_equal(one.cpu().numpy().reshape(m, -1), got[t:t + m]), t
    want = _ref(q, dk.cpu().numpy(), dv.cpu().numpy(), pos0)
    assert np.abs(got - want.reshape(n, -1)).max() / np.abs(want).max() < 1e-5


@pytest.mark.parametrize("hd,nkv", [(128, 8), (256, 4)])
def test_prefill_split_q8_kv_equals_decode(ctx, hd, nkv):
    """The same over a Q8_0 cache, where the prompt crosses into the wide chunks: the
    logits after a batched prompt equal those after the prompt token by token."""
    from hearth_amd import GGML_Q2_0, Model, ModelConfig
    cfg = ModelConfig(d_model=1024, n_layers=1, n_heads=2 * nkv, n_kv_heads=nkv, head_dim=hd, d_ffn=1024, vocab=512,
                      max_seq=2112, wtype=GGML_Q2_0, kv_type=8)
    toks = np.random.default_rng(hd).integers(0, 512, 40).tolist()
    got = []
    for batched in (True, False):
        m = Model(ctx, cfg)
        m.synthesize(3)
        m.prefill_kv_synthetic(4, 2030)
        if batched:
            m.prefill(toks[:-1], 2030)
        else:
            for i, t in enumerate(toks[:-1]):
                m.forward(t, 2030 + i, want_logits=False)
        got.append(m.forward(toks[-1], 2030 + len(toks) - 1)[0])
        m.close()
    assert np.array_equal(got[0], got[1])


@pytest.mark.parametrize("nh,nkv,hd,pos0", [
    (8, 8, 128, 62), (16, 8, 128, 2045), (24, 8, 128, 0), (32, 8, 128, 2043), (10, 2, 128, 500), (16, 2, 128, 8189),
    (4, 4, 256, 30), (8, 4, 256, 2046), (12, 4, 256, 3), (16, 4, 256, 2044), (24, 4, 256, 100), (16, 2, 256, 31),
    (8, 8, 256, 4200)])
def test_prefill_few_tokens_equal_decode(ctx, nh, nkv, hd, pos0):
    """1 to 10 tokens, on both sides of every line between the vector pass and the matrix
    form and across the narrow and wide chunks: each row equals hh_attention's bit for
    bit, with the cache's rows past the prompt not numbers."""
    rng = np.random.default_rng(nh * 100 + hd + pos0)
    top = 10
    ms = pos0 + top + 64
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()
    q = rng.standard_normal((top, nh, hd)).astype(np.float32)
    k = rng.standard_normal((nkv, ms, hd)).astype(np.float32) * 2
    v = rng.standard_normal((nkv, ms, hd)).astype(np.float32)
    dq, dk, dv = dev(q), dev(k), dev(v)
    print(f"prefill few tokens {nh}/{nkv} x {hd}, pos0 {pos0}", flush=True)
    want = []
    for t in range(top):
        one = torch.zeros(nh * hd, dtype=torch.float32, device="cuda")
        ctx.attention(dq[t].contiguous(), dk, dv, nh, nkv, hd, ms, pos0 + t + 1, one)
        ctx.sync()
        want.append(one.cpu().numpy())
    for n in range(top, 0, -1):
        dk[:, pos0 + n:] = float("nan")
        dv[:, pos0 + n:] = float("nan")
        out = torch.full((n * nh * hd + 64,), 7.0, dtype=torch.float32, device="cuda")
        ctx.attention_prefill(dq, dk, dv, nh, nkv, hd, ms, pos0, n, 0, out)
        ctx.sync()
        got = out.cpu().numpy()
        assert (got[n * nh * hd:] == 7.0).all()
        for t in range(n):
            assert np.array_equal(got[t * nh * hd:(t + 1) * nh * hd], want[t]), (n, t)


@pytest.mark.parametrize("nh,nkv,hd", [(16, 8, 128), (32, 8, 128), (16, 4, 256), (24, 4, 256)])
def test_prefill_few_tokens_q8_kv_equals_decode(ctx, nh, nkv, hd):
    """The same over a Q8_0 cache, through the batched prompt of a model: 3 tokens (the
    vector pass) and 12 (the matrix form) from a position where the chunks turn wide."""
    from hearth_amd import GGML_Q2_0, Model, ModelConfig
    cfg = ModelConfig(d_model=1024, n_layers=1, n_heads=nh, n_kv_heads=nkv, head_dim=hd, d_ffn=1024, vocab=512,
                      max_seq=2112, wtype=GGML_Q2_0, kv_type=8)
    m = Model(ctx, cfg)
    m.synthesize(3)
    for pos0 in (9, 2046):
        for n in (4, 13):
            toks = np.random.default_rng(n).integers(0, 512, n).tolist()
            got = []
            for batched in (True, False):
                m.prefill_kv_synthetic(4, pos0)
                if batched:
                    m.prefill(toks[:-1], pos0)
                else:
                    for i, t in enumerate(toks[:-1]):
                        m.forward(t, pos0 + i, want_logits=False)
                got.append(m.forward(toks[-1], pos0 + n - 1)[0])
            assert np.array_equal(got[0], got[1]), (pos0, n)
    m.close()


def _model_env(ctx, cfg, seed, env):
    from hearth_amd import Model
    old = os.environ.get("HH_PREFILL_ATTN")
    if env:
        os.environ["HH_PREFILL_ATTN"] = env
    else:
        os.environ.pop("HH_PREFILL_ATTN", None)
    try:
        m = Model(ctx, cfg)
    finally:
        if old is None:
            os.environ.pop("HH_PREFILL_ATTN", None)
        else:
            os.environ["HH_PREFILL_ATTN"] = old
    m.synthesize(seed)
    return m


@pytest.mark.parametrize("name,kv_type", [("9b-hybrid-q2", 0), ("8b-q2", 0), ("8b-q2", 8)])
def test_mfma_prefill_model_logits(ctx, oracle, name, kv_type):
    """The same prompt prefilled with the default attention and with the MFMA
    form: the first generated token's logits within 5e-2 relative (each
    regrouped sum can flip a later Q8_0 rounding, as the reference's own scalar
    and AVX2 arms do to each other)."""
    cfg = CONFIGS[name].replace(n_layers=2 if name == "8b-q2" else 8, max_seq=640, kv_type=kv_type)
    prompt = [oracle.synth_token(12, i, cfg.vocab) for i in range(300)]
    res = []
    for env in (None, "mfma"):
        m = _model_env(ctx, cfg, 41, env)
        m.prefill(prompt[:-1], 0)
        lg, _ = m.forward(prompt[-1], len(prompt) - 1)
        res.append(lg.astype(np.float64))
        m.close()
    err = float(np.abs(res[0] - res[1]).max() / np.abs(res[0]).max())
    print(f"{name} kv{kv_type}: logits rel err MFMA vs default prefill attention {err:.2e}", flush=True)
    assert np.isfinite(res[1]).all() and err < 5e-2, err


def test_attention_prefill_errors(ctx):
    from hearth_amd import HHError
    z = torch.zeros(16 * 4 * 128 * 64, dtype=torch.float32, device="cuda")
    cases = [((16, 4, 128, 64, 0, 16, 2), 1),      # mode
             ((16, 4, 128, 64, 60, 8, 0), 7),      # past max_seq
             ((16, 4, 96, 64, 0, 8, 1), 3),        # head_dim
             ((18, 1, 128, 64, 0, 8, 1), 3)]       # more than 8 query heads per kv head
    for (nh, nkv, hd, ms, pos0, n, mode), status in cases:
        with pytest.raises(HHError) as e:
            ctx.attention_prefill(z, z, z, nh, nkv, hd, ms, pos0, n, mode, z)
        assert e.value.status == status, (nh, nkv, hd, ms, pos0, n, mode, e.value)
