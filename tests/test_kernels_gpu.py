"""Parity of every HIP launcher with the CPU oracle on the same seeded inputs.

GPU results must be bit-identical to the oracle's GPU-order mode (same fp32 operations in the
same order) and within the parity tolerance of its exact mode: 1 bf16 ulp for RMSNorm,
RoPE and SwiGLU, bit-exact for the embedding rows, KV-cache slots and argmax. Shapes are the
Qwen3-0.6B decode layer (hidden 1024, 16q/8kv heads of 128, intermediate 3072, vocab 151936),
the Qwen3-4B widths (2560, 32/8, 9728) and the many-row roofline sweep sizes, plus ragged and
tiny edge cases."""
import math

import numpy as np
import pytest

from conftest import (bf16_bits, bf16_ulp_diff, bf16_vals, rand_bf16, ulp_bf16,
                      within_one_ulp_then_scale)

pytestmark = pytest.mark.gpu


def dev(bits):
    import torch
    return torch.from_numpy(np.ascontiguousarray(bits, dtype=np.uint16).view(np.int16)).cuda()


def host(t):
    import torch
    torch.cuda.synchronize()
    return t.cpu().numpy().view(np.uint16)


def dev_i32(a):
    import torch
    return torch.tensor(np.asarray(a, dtype=np.int32)).cuda()


def ident(name):
    print(f"[case] {name}", flush=True)


# ---------------------------------------------------------------- embedding

def test_embedding_rows_bit_exact(gpu, oracle):
    import torch
    ident("embedding 151936x1024 and 1000x2560")
    rng = np.random.default_rng(20)
    for vocab, hidden in [(151936, 1024), (1000, 2560), (50, 20)]:
        table = torch.randn(vocab, hidden, device="cuda").to(torch.bfloat16).view(torch.int16)
        for tok in [0, 1, vocab // 2, vocab - 1, int(rng.integers(0, vocab))]:
            out = torch.zeros(hidden, dtype=torch.int16, device="cuda")
            gpu.embedding_forward(out, table, dev_i32([tok]), hidden)
            assert np.array_equal(host(out), host(table[tok]))


# ---------------------------------------------------------------- RMSNorm

@pytest.mark.parametrize("rows,dim", [(1, 1024), (1, 2560), (4096, 2560), (3, 100), (2, 9000),
                                      (5, 8200), (7, 8192), (1, 8)])
def test_rmsnorm(gpu, oracle, rows, dim):
    ident(f"rmsnorm {rows}x{dim}")
    rng = np.random.default_rng(rows * 7 + dim)
    x = rand_bf16(rng, (rows, dim))
    w = rand_bf16(rng, dim, 0.1, 1.0)
    out = dev(np.zeros((rows, dim), np.uint16))
    gpu.rmsnorm_forward(out, dev(x), dev(w), rows, dim, 1e-6)
    y = host(out).reshape(rows, dim)
    assert np.array_equal(y, oracle.rmsnorm(x, w, 1e-6, oracle.GPU_ORDER))
    n_exact = oracle.rmsnorm(x, bf16_bits(np.ones(dim)), 1e-6, oracle.EXACT)
    assert within_one_ulp_then_scale(y, n_exact, w).all()


# one chunk and a tail, the last whole chunk of a wave, one to two waves (8192), two to five, the
# widest in chunks (131079) and the next row that is not; element offsets of the buffers
@pytest.mark.parametrize("dim", [7, 9, 15, 511, 513, 1023, 5000, 8191, 8193, 8200, 9001, 16384, 16391,
                                 32773, 131079, 131080])
@pytest.mark.parametrize("offset", [0, 1, 4])
def test_rmsnorm_row_forms(gpu, oracle, dim, offset):
    """Rows of any width at any element alignment, also in place, equal the oracle; the elements
    around the output stay."""
    import torch
    ident(f"rmsnorm rows of {dim} at element {offset}")
    rows = 5
    rng = np.random.default_rng(dim + offset)
    x, w = rand_bf16(rng, (rows, dim)), rand_bf16(rng, dim, 0.1, 1.0)
    pad = np.zeros(offset, np.uint16)
    xd = dev(np.concatenate([pad, x.reshape(-1), [0x7FC0] * 8]))
    wd = dev(np.concatenate([pad, w, [0x7FC0] * 8]))
    out = torch.full((offset + rows * dim + 8,), 0x1234, dtype=torch.int16, device="cuda")
    want = oracle.rmsnorm(x, w, 1e-6, oracle.GPU_ORDER).reshape(-1)
    gpu.rmsnorm_forward(out[offset:], xd[offset:], wd[offset:], rows, dim, 1e-6)
    got = host(out)
    assert np.array_equal(got[offset:offset + rows * dim], want)
    assert (got[:offset] == 0x1234).all() and (got[offset + rows * dim:] == 0x1234).all()
    gpu.rmsnorm_forward(xd[offset:], xd[offset:], wd[offset:], rows, dim, 1e-6)
    assert np.array_equal(host(xd)[offset:offset + rows * dim], want)


# ---------------------------------------------------------------- GEMV family

GEMV_SHAPES = [(4096, 1024), (1024, 2048), (1024, 3072), (2560, 9728), (2560, 4096),
               (151936, 1024), (37, 520), (5, 8), (3, 16400)]


@pytest.mark.parametrize("rows,cols", GEMV_SHAPES)
def test_gemv(gpu, oracle, rows, cols):
    ident(f"gemv {rows}x{cols}")
    rng = np.random.default_rng(rows + cols)
    w = rand_bf16(rng, (rows, cols), 0.02)
    x = rand_bf16(rng, cols)
    out = dev(np.zeros(rows, np.uint16))
    gpu.gemv_forward(out, dev(w), dev(x), rows, cols)
    y = host(out)
    assert np.array_equal(y, oracle.gemv(w, x, oracle.GPU_ORDER))
    # against exact arithmetic: one bf16 ulp after the single rounding, plus the fp32
    # accumulation bound 2 * cols * 2^-24 * sum|w x|
    wv, xv = bf16_vals(w).astype(np.float64), bf16_vals(x).astype(np.float64)
    exact = wv @ xv
    bound = ulp_bf16(exact) + 2 * cols * 2.0 ** -24 * (np.abs(wv) @ np.abs(xv))
    assert np.all(np.abs(bf16_vals(y) - exact) <= bound)


@pytest.mark.parametrize("rows,cols", [(1024, 2048), (1024, 3072), (2560, 4096), (2560, 9728),
                                       (33, 64)])
def test_gemv_residual(gpu, oracle, rows, cols):
    ident(f"gemv_residual {rows}x{cols}")
    rng = np.random.default_rng(rows * 3 + cols)
    w = rand_bf16(rng, (rows, cols), 0.02)
    inp = rand_bf16(rng, cols)
    x = rand_bf16(rng, rows)
    xd, tap = dev(x), dev(np.zeros(rows, np.uint16))
    gpu.gemv_residual_forward(xd, dev(w), dev(inp), rows, cols, tap)
    ex, et = oracle.gemv_residual(x, w, inp, oracle.GPU_ORDER, with_tap=True)
    assert np.array_equal(host(tap), et)
    assert np.array_equal(host(xd), ex)
    xd = dev(x)
    gpu.gemv_residual_forward(xd, dev(w), dev(inp), rows, cols, None)
    assert np.array_equal(host(xd), ex)


@pytest.mark.parametrize("hq,hkv,H", [(16, 8, 1024), (32, 8, 2560), (3, 1, 64)])
def test_qkv(gpu, oracle, hq, hkv, H):
    ident(f"qkv {hq}/{hkv} x {H}")
    rng = np.random.default_rng(hq + H)
    wq = rand_bf16(rng, (hq * 128, H), 0.02)
    wk = rand_bf16(rng, (hkv * 128, H), 0.02)
    wv = rand_bf16(rng, (hkv * 128, H), 0.02)
    x = rand_bf16(rng, H)
    q, k, v = (dev(np.zeros(n, np.uint16)) for n in (hq * 128, hkv * 128, hkv * 128))
    gpu.qkv_forward(q, k, v, dev(wq), dev(wk), dev(wv), dev(x), hq * 128, hkv * 128, H)
    eq, ek, ev = oracle.qkv(wq, wk, wv, x, oracle.GPU_ORDER)
    assert np.array_equal(host(q), eq)
    assert np.array_equal(host(k), ek)
    assert np.array_equal(host(v), ev)


@pytest.mark.parametrize("rows,cols", [(3072, 1024), (6144, 2048), (9728, 2560), (77, 136)])
def test_gate_up(gpu, oracle, rows, cols):
    ident(f"gate_up {rows}x{cols}")
    rng = np.random.default_rng(rows + 5 * cols)
    wg = rand_bf16(rng, (rows, cols), 0.02)
    wu = rand_bf16(rng, (rows, cols), 0.02)
    x = rand_bf16(rng, cols)
    act, gt, ut = (dev(np.zeros(rows, np.uint16)) for _ in range(3))
    gpu.gate_up_forward(act, dev(wg), dev(wu), dev(x), rows, cols, gt, ut)
    ea, eg, eu = oracle.gate_up(wg, wu, x, oracle.GPU_ORDER, with_taps=True)
    assert np.array_equal(host(gt), eg) and np.array_equal(host(ut), eu)
    assert np.array_equal(host(act), ea)
    s_exact = oracle.swiglu(eg, bf16_bits(np.ones(rows)), oracle.EXACT)
    assert within_one_ulp_then_scale(host(act), s_exact, eu).all()
    act2 = dev(np.zeros(rows, np.uint16))
    gpu.gate_up_forward(act2, dev(wg), dev(wu), dev(x), rows, cols, None, None)
    assert np.array_equal(host(act2), ea)


# ---------------------------------------------------------------- RMSNorm fused into the GEMV

FUSED_NORM_SHAPES = [(1024, 16, 8), (2560, 32, 8), (2048, 16, 8), (136, 3, 1),
                     (8192, 2, 1)]


@pytest.mark.parametrize("H,hq,hkv", FUSED_NORM_SHAPES)
def test_rmsnorm_fused_gemvs(gpu, oracle, H, hq, hkv):
    """The fused forms equal rmsnorm_forward followed by the plain launcher, bit for bit."""
    ident(f"rmsnorm fused qkv/gemv/gate_up H={H} {hq}/{hkv}")
    rng = np.random.default_rng(H + hq)
    x = rand_bf16(rng, H, 1.0, 4.0)
    g = rand_bf16(rng, H, 0.1, 1.0)
    xn = oracle.rmsnorm(x[None], g, 1e-6, oracle.GPU_ORDER)[0]
    wq = rand_bf16(rng, (hq * 128, H), 0.02)
    wk = rand_bf16(rng, (hkv * 128, H), 0.02)
    wv = rand_bf16(rng, (hkv * 128, H), 0.02)
    q, k, v = (dev(np.zeros(n, np.uint16)) for n in (hq * 128, hkv * 128, hkv * 128))
    gpu.rmsnorm_qkv_forward(q, k, v, dev(wq), dev(wk), dev(wv), dev(x), dev(g), 1e-6, hq * 128,
                            hkv * 128, H)
    eq, ek, ev = oracle.qkv(wq, wk, wv, xn, oracle.GPU_ORDER)
    assert np.array_equal(host(q), eq)
    assert np.array_equal(host(k), ek)
    assert np.array_equal(host(v), ev)
    rows = 3 * H + 5 if H <= 2560 else 1029
    w = rand_bf16(rng, (rows, H), 0.02)
    out = dev(np.zeros(rows, np.uint16))
    gpu.rmsnorm_gemv_forward(out, dev(w), dev(x), dev(g), 1e-6, rows, H)
    assert np.array_equal(host(out), oracle.gemv(w, xn, oracle.GPU_ORDER))
    wg = rand_bf16(rng, (rows, H), 0.02)
    act = dev(np.zeros(rows, np.uint16))
    gpu.rmsnorm_gate_up_forward(act, dev(wg), dev(w), dev(x), dev(g), 1e-6, rows, H)
    assert np.array_equal(host(act), oracle.gate_up(wg, w, xn, oracle.GPU_ORDER))


def test_rmsnorm_fused_gemv_rejects_wide_rows(gpu):
    """A row wider than 8192 columns is refused before any launch."""
    H = 8200
    x, g = dev(np.zeros(H, np.uint16)), dev(np.zeros(H, np.uint16))
    w = dev(np.zeros((4, H), np.uint16))
    out = dev(np.zeros(4, np.uint16))
    with pytest.raises(gpu.LlmError, match="do not fit one panel"):
        gpu.rmsnorm_gemv_forward(out, w, x, g, 1e-6, 4, H)


# ---------------------------------------------------------------- SwiGLU

@pytest.mark.parametrize("n", [65280, 4096 * 9728, 1001, 7])
def test_swiglu(gpu, oracle, n):
    ident(f"swiglu n={n}")
    rng = np.random.default_rng(n)
    if n == 65280:  # every finite bf16 gate value
        g = np.arange(65536, dtype=np.uint32).astype(np.uint16)
        g = g[np.isfinite(bf16_vals(g))]
    else:
        g = rand_bf16(rng, n, 2.0)
    u = rand_bf16(rng, g.size)
    act = dev(np.zeros(g.size, np.uint16))
    gpu.swiglu_forward(act, dev(g), dev(u), g.size)
    y = host(act)
    assert np.array_equal(y, oracle.swiglu(g, u, oracle.GPU_ORDER))
    s_exact = oracle.swiglu(g, bf16_bits(np.ones(g.size)), oracle.EXACT)
    assert within_one_ulp_then_scale(y, s_exact, u).all()
    if n == 65280:
        # u = 1: the rounded SiLU itself, for every finite bf16 gate value (the kernel's fast
        # estimate must round like the precise formula everywhere)
        ones = bf16_bits(np.ones(g.size))
        act1 = dev(np.zeros(g.size, np.uint16))
        gpu.swiglu_forward(act1, dev(g), dev(ones), g.size)
        assert np.array_equal(host(act1), oracle.swiglu(g, ones, oracle.GPU_ORDER))


# ---------------------------------------------------------------- QK-norm + RoPE + KV write

def rope_rotate(tap, positions, D, theta, oracle):
    """HF's apply_rotary_pos_emb on bf16 heads, computed independently: angles fp32(pos *
    inv_freq_j) (inv_freq pinned to decimal arithmetic), cos/sin from libm rounded through fp32
    to bf16, each product and the sum rounded to bf16 (modeling_qwen3.py:126-170)."""
    inv = oracle.inv_freq(theta, D)
    T = len(positions)
    y = bf16_vals(np.asarray(tap, dtype=np.uint16).reshape(T, -1, D))
    out = np.empty(y.shape, np.uint16)
    r = lambda z: bf16_vals(bf16_bits(z))
    for t, p in enumerate(positions):
        ang = (np.float32(p) * inv).astype(np.float32)
        c = bf16_vals(bf16_bits(np.array([math.cos(float(a)) for a in ang], np.float32)))
        s = bf16_vals(bf16_bits(np.array([math.sin(float(a)) for a in ang], np.float32)))
        a, b = y[t, :, :D // 2], y[t, :, D // 2:]
        out[t, :, :D // 2] = bf16_bits(r(a * c) - r(b * s))
        out[t, :, D // 2:] = bf16_bits(r(b * c) + r(a * s))
    return out


def _rope_case(rng, n_tokens, hq, hkv, D, max_seq):
    q = rand_bf16(rng, (n_tokens, hq * D))
    k = rand_bf16(rng, (n_tokens, hkv * D))
    v = rand_bf16(rng, (n_tokens, hkv * D))
    qn = rand_bf16(rng, D, 0.1, 1.0)
    kn = rand_bf16(rng, D, 0.1, 1.0)
    kc = np.full((max_seq, hkv * D), 0x7FC1, np.uint16)
    vc = np.full((max_seq, hkv * D), 0x7FC3, np.uint16)
    return q, k, v, qn, kn, kc, vc


@pytest.mark.parametrize("hq,hkv,D,pos", [(16, 8, 128, 0), (16, 8, 128, 1), (16, 8, 128, 3071),
                                          (32, 8, 128, 4095), (4, 2, 64, 77), (4, 2, 256, 500),
                                          (3, 1, 128, 9), (32, 8, 128, 4096), (32, 8, 128, 8191),
                                          (32, 8, 128, 8447)])
def test_qk_norm_rope_decode(gpu, oracle, hq, hkv, D, pos):
    """Config-1 decode: q/k rotated in place bit-exactly, k'/v written to cache row pos only.
    Positions past the reference's 4096-slot cap (src/forward.cu:7-8) use an 8448-slot cache, the
    size of the Qwen3-4B 8192-position config: the rows at 4096, 8191 and 8447 are written and
    every other row keeps its sentinel."""
    ident(f"qk_norm_rope decode {hq}/{hkv} D{D} pos{pos}")
    rng = np.random.default_rng(hq * 1000 + pos)
    max_seq = 4096 if pos < 4096 else 8448
    q, k, v, qn, kn, kc, vc = _rope_case(rng, 1, hq, hkv, D, max_seq)
    qd, kd, kcd, vcd = dev(q), dev(k), dev(kc), dev(vc)
    qt, kt = dev(np.zeros_like(q)), dev(np.zeros_like(k))
    gpu.qk_norm_rope_forward(qd, kd, dev(v), dev(qn), dev(kn), kcd, vcd, dev_i32([pos]), hq, hkv,
                             D, 1e-6, 1e6, qt, kt)
    eq, ek, ekc, evc, eqt, ekt = oracle.qk_norm_rope_rows(q, k, v, qn, kn, kc, vc, [pos], hq, hkv,
                                                          D, 1e-6, 1e6, oracle.GPU_ORDER,
                                                          with_taps=True)
    assert np.array_equal(host(qt).reshape(eqt.shape), eqt)
    assert np.array_equal(host(kt).reshape(ekt.shape), ekt)
    assert np.array_equal(host(qd).reshape(eq.shape), eq)
    assert np.array_equal(host(kd).reshape(ek.shape), ek)
    gkc, gvc = host(kcd).reshape(kc.shape), host(vcd).reshape(vc.shape)
    assert np.array_equal(gkc, ekc) and np.array_equal(gvc, evc)
    assert np.array_equal(gkc[pos], host(kd).reshape(-1)) and np.array_equal(gvc[pos], v[0])
    # tolerance against exact arithmetic: the normed heads within 1 ulp at HF's rounding point,
    # and the rotation of the GPU's own normed heads bit-exact against libm cos/sin
    ones = bf16_bits(np.ones(D))
    nq = oracle.qk_norm_rope_rows(q, k, v, ones, ones, kc, vc, [pos], hq, hkv, D, 1e-6, 1e6,
                                  oracle.EXACT, with_taps=True)
    assert within_one_ulp_then_scale(host(qt).reshape(-1), nq[4].reshape(-1), np.tile(qn, hq)).all()
    assert within_one_ulp_then_scale(host(kt).reshape(-1), nq[5].reshape(-1), np.tile(kn, hkv)).all()
    assert np.array_equal(host(qd).reshape(-1), rope_rotate(host(qt), [pos], D, 1e6, oracle).reshape(-1))
    assert np.array_equal(host(kd).reshape(-1), rope_rotate(host(kt), [pos], D, 1e6, oracle).reshape(-1))


def test_qk_norm_rope_rows_sweep(gpu, oracle):
    """Config-5 sweep: 4096 tokens x (32 q + 8 kv) heads of 128 at positions 0..4095."""
    ident("qk_norm_rope rows 4096 tokens 32/8")
    rng = np.random.default_rng(30)
    T, hq, hkv, D = 4096, 32, 8, 128
    q, k, v, qn, kn, kc, vc = _rope_case(rng, T, hq, hkv, D, T)
    pos = np.arange(T, dtype=np.int32)
    qd, kd, kcd, vcd = dev(q), dev(k), dev(kc), dev(vc)
    gpu.qk_norm_rope_rows(qd, kd, dev(v), dev(qn), dev(kn), kcd, vcd, dev_i32(pos), T, hq, hkv, D,
                          1e-6, 1e6)
    eq, ek, ekc, evc = oracle.qk_norm_rope_rows(q, k, v, qn, kn, kc, vc, pos, hq, hkv, D, 1e-6,
                                                1e6, oracle.GPU_ORDER)
    assert np.array_equal(host(qd).reshape(eq.shape), eq)
    assert np.array_equal(host(kd).reshape(ek.shape), ek)
    assert np.array_equal(host(kcd).reshape(kc.shape), ekc)
    assert np.array_equal(host(vcd).reshape(vc.shape), evc)


# ---------------------------------------------------------------- attention

@pytest.mark.parametrize("hq,hkv,pos", [(16, 8, 0), (16, 8, 4), (16, 8, 63), (16, 8, 64),
                                        (16, 8, 260), (32, 8, 4095), (32, 8, 8447), (8, 8, 100),
                                        (8, 1, 130), (3, 3, 4100)])
def test_attention(gpu, oracle, hq, hkv, pos):
    ident(f"attention {hq}/{hkv} pos{pos}")
    rng = np.random.default_rng(hq * 10000 + pos)
    D = 128
    max_seq = max(pos + 1, 4096) if pos < 8000 else 8448
    q = rand_bf16(rng, hq * D)
    kc = rand_bf16(rng, (max_seq, hkv * D))
    vc = rand_bf16(rng, (max_seq, hkv * D))
    import torch
    att = torch.zeros(gpu.attention_workspace_floats(hq, D, max_seq), dtype=torch.float32,
                      device="cuda")
    out = dev(np.zeros(hq * D, np.uint16))
    scale = float(np.float32(1.0 / np.sqrt(D)))
    gpu.attention_forward(out, dev(q), dev(kc), dev(vc), att, hq, hkv, D, dev_i32([pos]), max_seq,
                          scale)
    y = host(out)
    assert np.array_equal(y, oracle.attention(q, kc, vc, hq, hkv, D, pos, scale, oracle.GPU_ORDER))
    assert bf16_ulp_diff(y, oracle.attention(q, kc, vc, hq, hkv, D, pos, scale,
                                             oracle.EXACT)).max() <= 2


@pytest.mark.parametrize("D", [64, 256])
@pytest.mark.parametrize("rep", [1, 2, 4, 8])
def test_attention_head_dims(gpu, oracle, D, rep):
    """The head_dim 64 and 256 instantiations of the split-softmax kernels, for every GQA ratio
    they are built for, at a position that spans several 64-position blocks and ends inside one:
    bit-identical to the oracle's GPU order, within 2 bf16 ulps of exact arithmetic."""
    import torch
    hkv = 2
    hq, pos = hkv * rep, 200 + 37 * rep
    ident(f"attention D{D} rep{rep} pos{pos}")
    rng = np.random.default_rng(D * 100 + rep)
    max_seq = 512
    q = rand_bf16(rng, hq * D)
    kc = rand_bf16(rng, (max_seq, hkv * D))
    vc = rand_bf16(rng, (max_seq, hkv * D))
    att = torch.zeros(gpu.attention_workspace_floats(hq, D, max_seq), dtype=torch.float32,
                      device="cuda")
    out = dev(np.zeros(hq * D, np.uint16))
    scale = float(np.float32(1.0 / np.sqrt(D)))
    gpu.attention_forward(out, dev(q), dev(kc), dev(vc), att, hq, hkv, D, dev_i32([pos]), max_seq,
                          scale)
    y = host(out)
    assert np.array_equal(y, oracle.attention(q, kc, vc, hq, hkv, D, pos, scale, oracle.GPU_ORDER))
    assert bf16_ulp_diff(y, oracle.attention(q, kc, vc, hq, hkv, D, pos, scale,
                                             oracle.EXACT)).max() <= 2


# one item per kv head (nb = 1), PV and combine in one launch and in two, more than one staged chunk of
# partials (17000), and more items than a launch has workgroups (8200)
@pytest.mark.parametrize("hq,hkv,D,pos,max_seq", [
    (2, 2, 64, 5, 64), (16, 2, 64, 700, 704), (4, 4, 256, 127, 128), (8, 8, 64, 17000, 17001),
    (64, 8, 256, 8200, 8256), (8, 1, 128, 9000, 9001), (8, 8, 64, 1000, 65600), (4, 4, 128, -1, 200)])
def test_attention_one_launch_combine(gpu, oracle, hq, hkv, D, pos, max_seq):
    """The PV pass and the combine: bit-identical to the oracle whatever `att` held
    before (every bit set, another call's partials), at a later and an earlier
    position on the same workspace, and with NaN among the values. Position -1 (no history) gives
    zeros."""
    import torch
    ident(f"attention one-launch combine {hq}/{hkv} D{D} pos{pos} of {max_seq}")
    rng = np.random.default_rng(hq * 1000 + pos)
    kc = rand_bf16(rng, (max_seq, hkv * D))
    vc = rand_bf16(rng, (max_seq, hkv * D))
    floats = gpu.attention_workspace_floats(hq, D, max_seq)
    att = torch.full((floats,), -1, dtype=torch.int32, device="cuda").view(torch.float32)
    out = dev(np.full(hq * D, 0x1234, np.uint16))
    scale = float(np.float32(1.0 / np.sqrt(D)))
    kd, vd = dev(kc), dev(vc)
    for p in (pos, pos // 3, pos):
        q = rand_bf16(rng, hq * D)
        gpu.attention_forward(out, dev(q), kd, vd, att, hq, hkv, D, dev_i32([p]), max_seq, scale)
        want = (oracle.attention(q, kc, vc, hq, hkv, D, p, scale, oracle.GPU_ORDER) if p >= 0
                else np.zeros(hq * D, np.uint16))
        assert np.array_equal(host(out), want), p
    if pos < 0:
        return
    vc[pos // 2, 1], vc[pos // 2, 2] = 0xFFFF, 0x7FFF  # NaNs with every payload bit set
    gpu.attention_forward(out, dev(q), kd, dev(vc), att, hq, hkv, D, dev_i32([pos]), max_seq, scale)
    got, rep = host(out).copy(), hq // hkv
    nan = np.isnan(bf16_vals(got)).reshape(hq, D)
    assert nan[:rep, 1:3].all() and nan.sum() == 2 * rep
    got.reshape(hq, D)[:rep, 1:3] = want.reshape(hq, D)[:rep, 1:3]
    assert np.array_equal(got, want)


# histories around the combine's batches of blocks, and the longest that one launch takes; then two
# launches, just past each limit and around the batches of 16 and 256 blocks
@pytest.mark.parametrize("hq,hkv,D,max_seq,blocks", [
    (2, 2, 64, 6144, (1, 31, 32, 33, 64, 65, 95, 96)), (16, 8, 128, 6144, (32, 33, 64, 65, 96)),
    (2, 1, 256, 4096, (15, 16, 17, 32, 33, 64)), (4, 1, 256, 2048, (7, 8, 9, 16, 17, 32)),
    (16, 2, 256, 1024, (3, 4, 5, 8, 9, 16)),
    (16, 8, 128, 6145, (96, 97)), (16, 2, 256, 1025, (16, 17)), (16, 16, 64, 5121, (80, 81)),
    (2, 2, 64, 17408, (1, 15, 16, 17, 255, 256, 257, 272))])
def test_attention_combine_batches(gpu, oracle, hq, hkv, D, max_seq, blocks):
    """PV and combine in one launch and in two: bit-identical to the oracle at
    the first and the last position of each count of blocks, on one workspace that begins as ones."""
    import torch
    ident(f"attention combine batches {hq}/{hkv} D{D} of {max_seq}")
    rng = np.random.default_rng(hq * 10007 + max_seq)
    kc, vc = rand_bf16(rng, (max_seq, hkv * D)), rand_bf16(rng, (max_seq, hkv * D))
    kd, vd = dev(kc), dev(vc)
    floats = gpu.attention_workspace_floats(hq, D, max_seq)
    att = torch.full((floats,), -1, dtype=torch.int32, device="cuda").view(torch.float32)
    scale = float(np.float32(1.0 / np.sqrt(D)))
    for nb in blocks:
        for pos in {64 * nb - 64, min(64 * nb, max_seq) - 1}:
            q = rand_bf16(rng, hq * D)
            out = dev(np.full(hq * D, 0x1234, np.uint16))
            gpu.attention_forward(out, dev(q), kd, vd, att, hq, hkv, D, dev_i32([pos]), max_seq, scale)
            want = oracle.attention(q, kc, vc, hq, hkv, D, pos, scale, oracle.GPU_ORDER)
            assert np.array_equal(host(out), want), pos


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("max_seq", [200, 9000])  # PV and combine in one launch, and in two
def test_attention_position_outside_the_caches(gpu, fused, max_seq):
    """Positions the caches cannot hold: zeros, and no byte of the caches or the workspace, nor of what
    lies behind them, is written."""
    import torch
    ident(f"attention position outside {max_seq} fused {fused}")
    hq, hkv, D, behind = 4, 2, 128, 64
    g = torch.Generator(device="cuda").manual_seed(max_seq)
    x = [torch.randn(n, generator=g, device="cuda", dtype=torch.bfloat16)
         for n in (hq * D, hkv * D, hkv * D, D, D)]
    cache = torch.randn(2, max_seq + behind, hkv * D, generator=g, device="cuda", dtype=torch.bfloat16)
    floats = gpu.attention_workspace_floats(hq, D, max_seq)
    att = torch.randn(floats + behind * D * hq, generator=g, device="cuda")
    held = [cache.clone(), att.clone()]
    for pos in (max_seq, max_seq + 1, max_seq + 40, -1, -2, -200):
        out = torch.ones(hq * D, device="cuda", dtype=torch.bfloat16)
        if fused:
            gpu.qk_norm_rope_attention_forward(out, *x, cache[0], cache[1], att, dev_i32([pos]), hq, hkv,
                                               D, 1e-6, 1e6, max_seq, 0.1)
        else:
            gpu.attention_forward(out, x[0], cache[0], cache[1], att, hq, hkv, D, dev_i32([pos]), max_seq,
                                  0.1)
        torch.cuda.synchronize()
        assert not out.view(torch.int16).any(), pos  # +0 in every bit
        assert torch.equal(cache, held[0]) and torch.equal(att, held[1]), pos


@pytest.mark.parametrize("hq,hkv,D,max_seq", [(2, 2, 64, 640), (16, 8, 128, 640), (8, 1, 256, 640),
                                              (16, 8, 128, 9000)])
def test_attention_scores_not_numbers(gpu, oracle, hq, hkv, D, max_seq):
    """Scores that are NaN of every payload, or infinite, in all or the first blocks of a kv head (whose
    first block's max also counts the head's items where PV and combine are one launch): every output is
    written, NaN where the oracle's is and its bits elsewhere."""
    import torch
    ident(f"attention with scores that are not numbers {hq}/{hkv} D{D} of {max_seq}")
    rng = np.random.default_rng(hq + D)
    pos, scale = 600, float(np.float32(1.0 / np.sqrt(D)))
    q, kc, vc = rand_bf16(rng, hq * D), rand_bf16(rng, (max_seq, hkv * D)), rand_bf16(rng, (max_seq, hkv * D))
    att = torch.zeros(gpu.attention_workspace_floats(hq, D, max_seq), device="cuda")
    for bits in (0xFFFF, 0x7FFF, 0x7F81, 0xFF81, 0x7FC0, 0x7F80, 0xFF80):
        for rows in (slice(0, max_seq), slice(0, 64), slice(0, 1), slice(64, 128)):
            keys = kc.copy()
            keys[rows, :D] = bits  # the first kv head's
            out = dev(np.full(hq * D, 0x1234, np.uint16))
            gpu.attention_forward(out, dev(q), dev(keys), dev(vc), att, hq, hkv, D, dev_i32([pos]), max_seq,
                                  scale)
            want = oracle.attention(q, keys, vc, hq, hkv, D, pos, scale, oracle.GPU_ORDER)
            got, nan = host(out), np.isnan(bf16_vals(want))
            assert np.array_equal(got[~nan], want[~nan]), (hex(bits), rows)
            assert np.isnan(bf16_vals(got)[nan]).all(), (hex(bits), rows)


# the shapes whose last blocks' workgroups are the most and the largest
@pytest.mark.parametrize("hq,hkv,D,max_seq", [(64, 8, 128, 2048), (64, 8, 256, 1024), (64, 8, 128, 8192),
                                              (32, 8, 256, 2048)])
def test_attention_overlapping_streams(gpu, hq, hkv, D, max_seq):
    """Attention calls of both forms on six streams at once, each with a workspace of its own: every
    result is that of the same call alone."""
    import torch
    ident(f"attention on six streams {hq}/{hkv} D{D} of {max_seq}")
    g = torch.Generator(device="cuda").manual_seed(hq + D + max_seq)
    bf = torch.bfloat16

    def normal(*shape):
        return torch.randn(*shape, generator=g, device="cuda", dtype=bf)

    scale, kvd, n = float(np.float32(1.0 / np.sqrt(D))), hkv * D, 6
    kc, vc, norm = normal(max_seq, kvd), normal(max_seq, kvd), normal(D)
    own = [dict(q=normal(hq * D), k=normal(kvd), v=normal(kvd), kc=kc.clone(), vc=vc.clone(),
                att=torch.empty(gpu.attention_workspace_floats(hq, D, max_seq), device="cuda"),
                pos=dev_i32([max_seq - 1 - 100 * i]), out=torch.zeros(4, hq * D, device="cuda", dtype=bf))
           for i in range(n)]

    def call(c, i, row, stream):
        if i % 2:
            gpu.qk_norm_rope_attention_forward(c["out"][row], c["q"], c["k"], c["v"], norm, norm,
                                               c["kc"], c["vc"], c["att"], c["pos"], hq, hkv, D, 1e-6,
                                               1e6, max_seq, scale, stream=stream)
        else:
            gpu.attention_forward(c["out"][row], c["q"], c["kc"], c["vc"], c["att"], hq, hkv, D,
                                  c["pos"], max_seq, scale, stream=stream)

    torch.cuda.synchronize()
    for i, c in enumerate(own):
        call(c, i, 0, None)
        torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(n)]
    for row in range(1, 4):
        for i, c in enumerate(own):
            call(c, i, row, streams[i])
    torch.cuda.synchronize()
    for c in own:
        rows = c["out"].view(torch.int16)
        assert c["out"][0].isfinite().all() and c["out"][0].any()
        for row in range(1, 4):
            assert torch.equal(rows[0], rows[row])


@pytest.mark.parametrize("hq,hkv,D", [(8, 1, 64), (2, 1, 128), (4, 1, 128), (1, 1, 256)])
def test_attention_statistics_chunks(gpu, oracle, hq, hkv, D):
    """Histories around 1 to 4 chunks of 64 block statistics, and past them, equal the oracle; with
    scores so far apart that whole blocks weigh nothing, and infinite keys."""
    import torch
    ident(f"attention statistics {hq}/{hkv} D{D}")
    rng = np.random.default_rng(hq * D)
    max_seq = 16448
    kc, vc = rand_bf16(rng, (max_seq, hkv * D)), rand_bf16(rng, (max_seq, hkv * D))
    far = kc.copy()
    far[4000:9000] = rand_bf16(rng, (5000, hkv * D), 40.0)
    inf = kc.copy()
    inf[5000, 3] = 0x7F80
    att = torch.zeros(gpu.attention_workspace_floats(hq, D, max_seq), device="cuda")
    scale = float(np.float32(1.0 / np.sqrt(D)))
    vd = dev(vc)
    for keys in (kc, far, inf):
        kd = dev(keys)
        for pos in (4095, 4096, 8191, 8192, 12287, 12288, 16383, 16384):
            q = rand_bf16(rng, hq * D)
            out = dev(np.zeros(hq * D, np.uint16))
            gpu.attention_forward(out, dev(q), kd, vd, att, hq, hkv, D, dev_i32([pos]), max_seq, scale)
            want = oracle.attention(q, keys, vc, hq, hkv, D, pos, scale, oracle.GPU_ORDER)
            got, nan = host(out), np.isnan(bf16_vals(want))
            assert np.array_equal(got[~nan], want[~nan]), pos
            assert np.isnan(bf16_vals(got)[nan]).all(), pos


FUSED_ATTN_CASES = [(16, 8, 128, 0, 4096), (16, 8, 128, 63, 4096), (16, 8, 128, 64, 4096),
                    (16, 8, 128, 260, 4096), (32, 8, 128, 8192, 8448), (32, 8, 128, 8447, 8448),
                    (8, 8, 128, 100, 512), (8, 1, 128, 130, 512), (2, 2, 64, 301, 512),
                    (16, 2, 64, 200, 512), (4, 2, 256, 777, 1024), (16, 2, 256, 150, 512),
                    (3, 3, 128, 4100, 4200)]


@pytest.mark.parametrize("hq,hkv,D,pos,max_seq", FUSED_ATTN_CASES)
def test_qk_norm_rope_attention_fused(gpu, oracle, hq, hkv, D, pos, max_seq):
    """qk_norm_rope_attention_forward (QK-norm + RoPE inside the attention's scores pass): the
    output is bit-identical to the oracle's GPU order of the two steps (QK-norm + RoPE of q and
    k, k'/v written to row pos, then attention over rows 0..pos), the caches equal the oracle's
    (row pos written, every other row keeps its value), q and k are not rewritten. Three calls
    on one workspace: the case, an earlier position with new inputs, then the first position
    again with new inputs."""
    import torch
    ident(f"qk_norm_rope_attention {hq}/{hkv} D{D} pos{pos} max_seq{max_seq}")
    rng = np.random.default_rng(hq * 7919 + hkv * 31 + D + pos)
    kc = rand_bf16(rng, (max_seq, hkv * D))
    vc = rand_bf16(rng, (max_seq, hkv * D))
    kcd, vcd = dev(kc), dev(vc)
    att = torch.zeros(gpu.attention_workspace_floats(hq, D, max_seq), dtype=torch.float32,
                      device="cuda")
    scale = float(np.float32(1.0 / np.sqrt(D)))
    qn = rand_bf16(rng, D, 0.1, 1.0)
    kn = rand_bf16(rng, D, 0.1, 1.0)
    for p in [pos, pos // 2, pos]:
        q = rand_bf16(rng, hq * D)
        k = rand_bf16(rng, hkv * D)
        v = rand_bf16(rng, hkv * D)
        qd, kd = dev(q), dev(k)
        out = dev(np.zeros(hq * D, np.uint16))
        gpu.qk_norm_rope_attention_forward(out, qd, kd, dev(v), dev(qn), dev(kn), kcd, vcd, att,
                                           dev_i32([p]), hq, hkv, D, 1e-6, 1e6, max_seq, scale)
        eq, ek, ekc, evc = oracle.qk_norm_rope_rows(q[None], k[None], v[None], qn, kn, kc, vc, [p],
                                                    hq, hkv, D, 1e-6, 1e6, oracle.GPU_ORDER)
        want = oracle.attention(eq.reshape(-1), ekc, evc, hq, hkv, D, p, scale, oracle.GPU_ORDER)
        got = host(out)
        assert np.array_equal(got, want), p
        assert np.array_equal(host(kcd).reshape(kc.shape), ekc), p
        assert np.array_equal(host(vcd).reshape(vc.shape), evc), p
        assert np.array_equal(host(qd), q) and np.array_equal(host(kd), k)
        kc, vc = ekc, evc


ONE_PASS_CASES = [(16, 8, 128, 0, 4096), (16, 8, 128, 63, 4096), (16, 8, 128, 64, 4096),
                  (16, 8, 128, 260, 4096), (16, 8, 128, 4095, 4096), (32, 8, 128, 8192, 8448),
                  (32, 8, 128, 8447, 8448), (32, 8, 128, 30001, 32768), (8, 8, 128, 100, 512),
                  (8, 1, 128, 130, 512), (8, 1, 128, 9000, 9100), (2, 2, 128, 301, 512),
                  (16, 2, 128, 2000, 2048), (3, 3, 128, 4100, 4200)]


@pytest.mark.parametrize("hq,hkv,D,pos,max_seq", ONE_PASS_CASES)
def test_qk_norm_rope_attention_one_pass(gpu, oracle, hq, hkv, D, pos, max_seq):
    """qk_norm_rope_attention_one_pass (QK-norm + RoPE + attention in one launch, the
    workgroups of a kv head handing block statistics and partial outputs to each other): the
    output is bit-identical to the oracle's GPU order of the two steps, the caches equal the
    oracle's (row pos written, every other row unchanged), q and k are not rewritten and the
    error flag stays 0. Five calls on one workspace (its launch counter tags the handoffs): the
    case, an earlier position, the case again, the first position and the case once more, each
    with new inputs, so a stale word of an earlier call would be read as current."""
    import torch
    if not gpu.attention_one_pass_supported(hq, hkv, D, max_seq):
        pytest.skip("no one-pass attention for this shape on this device")
    ident(f"one-pass attention {hq}/{hkv} D{D} pos{pos} max_seq{max_seq}")
    rng = np.random.default_rng(hq * 7919 + hkv * 31 + D + pos + 17)
    kc = rand_bf16(rng, (max_seq, hkv * D))
    vc = rand_bf16(rng, (max_seq, hkv * D))
    kcd, vcd = dev(kc), dev(vc)
    ws = torch.zeros(gpu.attention_one_pass_bytes(hq, D, max_seq), dtype=torch.uint8,
                     device="cuda")
    err = dev_i32([0])
    scale = float(np.float32(1.0 / np.sqrt(D)))
    qn = rand_bf16(rng, D, 0.1, 1.0)
    kn = rand_bf16(rng, D, 0.1, 1.0)
    for p in [pos, pos // 2, pos, 0, pos]:
        q = rand_bf16(rng, hq * D)
        k = rand_bf16(rng, hkv * D)
        v = rand_bf16(rng, hkv * D)
        qd, kd = dev(q), dev(k)
        out = dev(np.zeros(hq * D, np.uint16))
        gpu.qk_norm_rope_attention_one_pass(out, qd, kd, dev(v), dev(qn), dev(kn), kcd, vcd, ws,
                                            err, dev_i32([p]), hq, hkv, D, 1e-6, 1e6, max_seq,
                                            scale)
        eq, ek, ekc, evc = oracle.qk_norm_rope_rows(q[None], k[None], v[None], qn, kn, kc, vc, [p],
                                                    hq, hkv, D, 1e-6, 1e6, oracle.GPU_ORDER)
        want = oracle.attention(eq.reshape(-1), ekc, evc, hq, hkv, D, p, scale, oracle.GPU_ORDER)
        got = host(out)
        assert int(err.cpu()[0]) == 0, p
        assert np.array_equal(got, want), p
        assert np.array_equal(host(kcd).reshape(kc.shape), ekc), p
        assert np.array_equal(host(vcd).reshape(vc.shape), evc), p
        assert np.array_equal(host(qd), q) and np.array_equal(host(kd), k)
        kc, vc = ekc, evc


def test_qk_norm_rope_attention_one_pass_rejects(gpu):
    """Shapes the one-pass attention is not built for are refused with a message, and report
    themselves as unsupported."""
    import torch
    ws = torch.zeros(1 << 20, dtype=torch.uint8, device="cuda")
    x = dev(np.zeros(4096, np.uint16))
    err = dev_i32([0])
    for hq, hkv, D, max_seq in [(4, 2, 64, 16), (6, 2, 128, 16), (16, 8, 128, 40000)]:
        assert not gpu.attention_one_pass_supported(hq, hkv, D, max_seq)
        with pytest.raises(gpu.LlmError):
            gpu.qk_norm_rope_attention_one_pass(x, x, x, x, x, x, x, x, ws, err, dev_i32([0]), hq,
                                                hkv, D, 1e-6, 1e6, max_seq, 0.1)
    with pytest.raises(gpu.LlmError):  # no norm weights
        gpu.qk_norm_rope_attention_one_pass(x, x, x, x, None, None, x, x, ws, err, dev_i32([0]),
                                            4, 2, 128, 1e-6, 1e6, 16, 0.1)


def test_attention_rejects_a_workspace_too_small(gpu):
    """The C-ABI guard on `att`: a workspace sized for fewer positions than max_seq (here a
    RunState's own att, allocated for 64 positions, passed with max_seq 4096, as a caller sizing
    it [n_heads, max_seq] the reference's way would under-size it) is an error, not an overrun;
    the same buffer at its own size runs."""
    from llm_inference_amd import model
    cfg = model.make_config(hidden_size=512, intermediate_size=1024, n_layers=1, n_heads=8,
                            n_kv_heads=4, vocab_size=256, max_seq_len=64)
    dec = model.Decoder(cfg, ("synth", 1, 0.02, 0.1))
    try:
        D, hq, hkv = 128, 8, 4
        q = dev(np.zeros(hq * D, np.uint16))
        kc = dev(np.zeros((4096, hkv * D), np.uint16))
        out = dev(np.zeros(hq * D, np.uint16))
        att = int(dec.s.att)
        with pytest.raises(gpu.LlmError, match="att has room"):
            gpu.attention_forward(out, q, kc, kc, att, hq, hkv, D, dev_i32([10]), 4096, 0.1)
        gpu.attention_forward(out, q, kc, kc, att, hq, hkv, D, dev_i32([10]), 64, 0.1)
        host(out)
    finally:
        dec.close()


@pytest.mark.parametrize("hq,hkv,pos,max_seq", [(32, 8, 8447, 8448), (16, 8, 4095, 4096),
                                                 (16, 8, 300, 4096)])
def test_attention_reference_sized_att(gpu, oracle, hq, hkv, pos, max_seq):
    """attention_forward with `att` allocated the reference's way (src/forward.cu:10-51: its own
    hipMalloc of [n_heads, max_seq] floats, src/forward.cuh:13): the scores go there and the
    block statistics and partial outputs to the library's own array. Bit-identical to the
    oracle's GPU order; a call with the full workspace in between leaves the next reference-sized
    call unaffected (every value it reads it wrote)."""
    import ctypes
    import torch
    from llm_inference_amd import model
    ident(f"attention reference-sized att {hq}/{hkv} pos{pos}")
    rt = model._hip()
    D = 128
    nbytes = hq * max_seq * 4
    ptr = ctypes.c_void_p()
    assert rt.hipMalloc(ctypes.byref(ptr), ctypes.c_size_t(nbytes)) == 0
    try:
        base, size = ctypes.c_void_p(), ctypes.c_size_t()
        assert rt.hipMemGetAddressRange(ctypes.byref(base), ctypes.byref(size), ptr) == 0
        full = gpu.attention_workspace_floats(hq, D, max_seq) * 4
        print(f"[case] att allocation {size.value} bytes; the full workspace needs {full}",
              flush=True)
        if (hq, max_seq) == (32, 8448):
            assert size.value < full  # this case runs on the library's array
        rng = np.random.default_rng(hq * 1000 + pos)
        scale = float(np.float32(1.0 / np.sqrt(D)))
        for rnd in range(2):
            q = rand_bf16(rng, hq * D)
            kc = rand_bf16(rng, (max_seq, hkv * D))
            vc = rand_bf16(rng, (max_seq, hkv * D))
            qd, kd, vd = dev(q), dev(kc), dev(vc)
            out = dev(np.full(hq * D, 0x7FC1, np.uint16))
            gpu.attention_forward(out, qd, kd, vd, ptr.value, hq, hkv, D, dev_i32([pos]),
                                  max_seq, scale)
            assert np.array_equal(host(out), oracle.attention(q, kc, vc, hq, hkv, D, pos, scale,
                                                              oracle.GPU_ORDER)), rnd
            if rnd == 0:  # the full-workspace form in between, on other data
                att = torch.zeros(full // 4, dtype=torch.float32, device="cuda")
                gpu.attention_forward(out, dev(rand_bf16(rng, hq * D)), kd, vd, att, hq, hkv, D,
                                      dev_i32([pos // 2]), max_seq, scale)
                host(out)
    finally:
        torch.cuda.synchronize()
        rt.hipFree(ptr)


def test_qk_norm_rope_attention_fused_rejects(gpu):
    """Shapes the kernels are not built for are refused with a message."""
    import torch
    att = torch.zeros(1 << 16, dtype=torch.float32, device="cuda")
    x = dev(np.zeros(4096, np.uint16))
    with pytest.raises(gpu.LlmError):  # head_dim 96
        gpu.qk_norm_rope_attention_forward(x, x, x, x, x, x, x, x, att, dev_i32([0]), 4, 2, 96,
                                           1e-6, 1e6, 16, 0.1)
    with pytest.raises(gpu.LlmError):  # 3 query heads per kv head
        gpu.qk_norm_rope_attention_forward(x, x, x, x, x, x, x, x, att, dev_i32([0]), 6, 2, 128,
                                           1e-6, 1e6, 16, 0.1)
    with pytest.raises(gpu.LlmError):  # no norm weights
        gpu.qk_norm_rope_attention_forward(x, x, x, x, None, None, x, x, att, dev_i32([0]), 4, 2,
                                           128, 1e-6, 1e6, 16, 0.1)


def test_hbm_stream_probe(gpu):
    """The ceiling probe's three modes compute what they claim (copy, xor of two streams, and a
    per-thread xor of the read chunks), including a length that is not a multiple of the grid."""
    import torch
    ident("hbm_stream_probe")
    n16 = 1024 * 256 * 4 * 3 + 5  # grid-stride remainder for the read mode
    a = torch.randint(0, 1 << 30, (n16 * 4,), dtype=torch.int32, device="cuda")
    b = torch.randint(0, 1 << 30, (n16 * 4,), dtype=torch.int32, device="cuda")
    dst = torch.zeros(n16 * 4, dtype=torch.int32, device="cuda")
    gpu.hbm_stream_probe(dst, a, None, n16 * 16, 1)
    assert torch.equal(dst, a)
    gpu.hbm_stream_probe(dst, a, b, n16 * 16, 2)
    assert torch.equal(dst, a ^ b)
    out = torch.zeros(1 << 18, dtype=torch.int32, device="cuda")
    gpu.hbm_stream_probe(out, a, None, n16 * 16, 0)
    # thread b * 256 + i xors chunks b * 1024 + i + 256 u + (1024 * 1024) j (all four words)
    chunks = a.view(n16, 4).cpu().numpy().astype(np.uint32)
    words = np.bitwise_xor.reduce(chunks, axis=1)
    c = np.arange(n16) % (1024 * 1024)
    thread = (c // 1024) * 256 + c % 256
    expect = np.zeros(1 << 18, np.uint32)
    np.bitwise_xor.at(expect, thread, words)
    assert np.array_equal(out.cpu().numpy().astype(np.uint32), expect)


def test_hbm_read_peak_probe(gpu):
    """The read-peak probe reads every chunk of its walk: a buffer of zeros with the magic word in
    one chunk of a late round (grid-stride: thread 5, third pass, last load; one range per
    workgroup: workgroup 1's thread 5, third pass, last load) makes exactly that thread store
    it; without it nothing is stored. Every loads-in-flight count and both layouts, with a
    length that is not a multiple of the grid; bad launch shapes are refused."""
    import torch
    ident("hbm_read_peak_probe")
    magic = 0x9e3779b9 - (1 << 32)  # as int32
    for contiguous in (0, 1):
        for U in (4, 8, 16):
            for blocks, threads in [(3, 256), (2, 1024), (7, 64)]:
                T = blocks * threads
                if contiguous:
                    span = U * threads * 3
                    n16 = blocks * span - 5  # the last workgroup's range is short
                    hit = span + U * threads * 2 + (U - 1) * threads + 5
                else:
                    n16 = U * T * 3 + 7
                    hit = U * T * 2 + (U - 1) * T + 5
                a = torch.zeros(n16 * 4, dtype=torch.int32, device="cuda")
                out = torch.zeros(1, dtype=torch.int32, device="cuda")
                gpu.hbm_read_peak_probe(out, a, n16 * 16, blocks, threads, U, contiguous)
                torch.cuda.synchronize()
                assert int(out.item()) == 0, (contiguous, U, blocks, threads)
                a[4 * hit] = magic
                gpu.hbm_read_peak_probe(out, a, n16 * 16, blocks, threads, U, contiguous)
                torch.cuda.synchronize()
                assert int(out.item()) == magic, (contiguous, U, blocks, threads)
    with pytest.raises(gpu.LlmError):
        gpu.hbm_read_peak_probe(out, a, 64, 4, 100)
    with pytest.raises(gpu.LlmError):
        gpu.hbm_read_peak_probe(out, a, 24, 4, 256)
    with pytest.raises(gpu.LlmError):
        gpu.hbm_read_peak_probe(out, a, 64, 4, 256, 6)
    with pytest.raises(gpu.LlmError):
        gpu.hbm_read_peak_probe(out, a, 64, 4, 256, 4, 2)


def test_hbm_copy_peak_probe(gpu):
    """The copy-peak probe copies every chunk exactly once and nothing past n_bytes: random words
    into a destination filled with a sentinel one chunk longer, for every chunks-in-flight count,
    with lengths that are not multiples of the grid's tile; bad launch shapes are refused."""
    import torch
    ident("hbm_copy_peak_probe")
    g = torch.Generator(device="cpu").manual_seed(11)
    for U in (1, 2, 4, 8):
        for blocks, threads in [(3, 256), (2, 1024), (7, 64)]:
            n16 = U * blocks * threads * 3 + 5
            a = torch.randint(-2**31, 2**31 - 1, (n16 * 4,), generator=g, dtype=torch.int32).cuda()
            d = torch.full((n16 * 4 + 4,), 0x5a5a5a5a, dtype=torch.int32, device="cuda")
            gpu.hbm_copy_peak_probe(d, a, n16 * 16, blocks, threads, U)
            torch.cuda.synchronize()
            assert torch.equal(d[:n16 * 4], a), (U, blocks, threads)
            assert torch.all(d[n16 * 4:] == 0x5a5a5a5a), (U, blocks, threads)
    with pytest.raises(gpu.LlmError):
        gpu.hbm_copy_peak_probe(d, a, 64, 4, 100)
    with pytest.raises(gpu.LlmError):
        gpu.hbm_copy_peak_probe(d, a, 24, 4, 256)
    with pytest.raises(gpu.LlmError):
        gpu.hbm_copy_peak_probe(d, a, 64, 4, 256, 3)


# ---------------------------------------------------------------- exponential

def test_exp_forms_agree_for_every_float(gpu, oracle):
    """The device's exponential without branches and with early returns: the same bits for each of the
    2^32 fp32 inputs (both zeros, infinities, denormals and every NaN among them), and the oracle's on
    a sample of them and around the limits of the clamp and the early returns."""
    import ctypes
    import torch
    ident("exp_f32 over every fp32 input")
    fn = gpu.lib().llm_exp_bits
    fn.argtypes = [ctypes.c_void_p, ctypes.c_uint32, ctypes.c_uint32, ctypes.c_int, ctypes.c_void_p]
    fn.restype = None
    stream = torch.cuda.current_stream().cuda_stream
    chunk = 1 << 28
    a, b = (torch.empty(chunk, dtype=torch.int32, device="cuda") for _ in range(2))
    rng = np.random.default_rng(104)
    edges = np.float32([-105, -104, -103.97, -87.3, 0, 88.72, 88.73, 89, 90, np.inf, -np.inf])
    edges = (edges.view(np.uint32)[:, None].astype(np.int64) + np.arange(-40, 41)).reshape(-1)
    bits = np.unique(np.concatenate([edges, rng.integers(0, 1 << 32, 20000)]) & 0xFFFFFFFF)
    for first in range(0, 1 << 32, chunk):
        for t, branches in ((a, 0), (b, 1)):
            fn(t.data_ptr(), first, chunk, branches, stream)
        assert torch.equal(a, b), hex(first)
        some = bits[(bits >= first) & (bits < first + chunk)]
        got = a[torch.from_numpy(some - first).cuda()].cpu().numpy().view(np.float32)
        x = some.astype(np.uint32).view(np.float32)
        want = np.float32([oracle.exp_f32(v) for v in x])
        nan = np.isnan(x)
        assert np.array_equal(got.view(np.uint32)[~nan], want.view(np.uint32)[~nan])
        assert np.isnan(got[nan]).all()
    gpu.check()


# ---------------------------------------------------------------- temperature sampling

def test_sample_forward(gpu, oracle):
    """sample_forward equals the oracle's inverse-CDF draw (same weights, same order of additions)
    on random rows, one-hot rows and uniform rows, for several temperatures and coins."""
    import torch
    ident("sample_forward")
    rng = np.random.default_rng(11)
    out = torch.zeros(1, dtype=torch.int32, device="cuda")
    n = 151936
    rows = [rand_bf16(rng, n, s) for s in (0.5, 2.0, 4.0)]
    hot = bf16_bits(np.full(n, -50.0, np.float32))
    hot[123456] = bf16_bits(np.array([50.0], np.float32))[0]
    rows += [hot, bf16_bits(np.zeros(n, np.float32)), rand_bf16(rng, 1000, 1.0),
             rand_bf16(rng, 1023, 1.0)]
    for row in rows:
        xd = dev(row)
        for inv_temp in (1.0, 0.7, 1.5):
            for u in (0.0, 0.25, 0.5, 0.9, 0.999):
                gpu.sample_forward(out, xd, row.size, inv_temp, u)
                assert int(out.item()) == oracle.sample(row, inv_temp, u), (row.size, inv_temp, u)


# chunk lengths around the staged piece (256 weights), rows around the one-launch limit (12288)
@pytest.mark.parametrize("n", [1, 16, 1025, 12288, 12289, 16 * 1024 + 1, 262144, 262145, 300001])
def test_sample_forward_row_lengths(gpu, oracle, n):
    """Both forms of the draw (one launch; sums spread over workgroups, drawn by the last) equal the
    oracle: random rows, a row that is mostly -inf, rows with a NaN and an inf, an unaligned view."""
    import torch
    ident(f"sample_forward row of {n}")
    rng = np.random.default_rng(n)
    out = torch.zeros(1, dtype=torch.int32, device="cuda")
    sparse = np.full(n, 0xFF80, np.uint16)  # -inf
    sparse[rng.integers(0, n, 5)] = rand_bf16(rng, 5)
    nan, inf = rand_bf16(rng, n), rand_bf16(rng, n)
    nan[n // 2], inf[n // 3] = 0x7FC0, 0x7F80
    for row in (rand_bf16(rng, n, 2.0), sparse, nan, inf):
        xd = dev(np.concatenate([row[:1], row]))
        for x in (dev(row), xd[1:]):
            for inv_temp, u in ((1.0, 0.0), (0.7, 0.4), (2.5, 0.9999)):
                gpu.sample_forward(out, x, n, inv_temp, u)
                assert int(out.item()) == oracle.sample(row, inv_temp, u), (inv_temp, u)


def test_sample_forward_overlapping_streams_and_graph(gpu, oracle):
    """Draws in flight on six streams at once, and a captured draw replayed between eager ones, each
    equal to the oracle: calls share nothing but the library's slots."""
    import torch
    ident("sample_forward on six streams and in a graph")
    rng = np.random.default_rng(77)
    n, coins = 151936, [float(c) for c in rng.random(8)]
    rows = [rand_bf16(rng, n, 2.0) for _ in range(6)]
    xs = [dev(r) for r in rows]
    outs = torch.full((6, 8), -7, dtype=torch.int32, device="cuda")
    streams = [torch.cuda.Stream() for _ in range(6)]
    want = [[oracle.sample(r, 0.8, c) for c in coins] for r in rows]
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(streams[0]):
        graph.capture_begin()
        gpu.sample_forward(outs[0, 0:], xs[0], n, 0.8, coins[0])
        graph.capture_end()
    for _ in range(3):
        outs.fill_(-7)
        torch.cuda.synchronize()
        for j, c in enumerate(coins):
            for i, s in enumerate(streams):
                if (i, j) != (0, 0):
                    gpu.sample_forward(outs[i, j:], xs[i], n, 0.8, c, stream=s)
        graph.replay()
        torch.cuda.synchronize()
        assert outs.cpu().tolist() == want


@pytest.mark.parametrize("n", [12289, 151936])
def test_sample_forward_with_every_slot_taken(gpu, oracle, n):
    """A call that finds its slot taken draws in its first launch; slots given back serve again."""
    import torch
    ident(f"sample_forward without slots, row of {n}")
    rng = np.random.default_rng(n)
    row = rand_bf16(rng, n, 2.0)
    xd, out = dev(row), torch.zeros(1, dtype=torch.int32, device="cuda")
    coins = [float(c) for c in rng.random(4)]
    want = [oracle.sample(row, 0.8, c) for c in coins]
    for taken in (1, 0):
        torch.cuda.synchronize()
        assert gpu.lib().llm_sample_slots(taken) == 0
        for c, w in zip(coins, want):
            gpu.sample_forward(out, xd, n, 0.8, c)
            assert int(out.item()) == w
        assert gpu.lib().llm_sample_slots(0) == (64 if taken else 0)


def test_sample_forward_shared_out(gpu, oracle):
    """Overlapping calls that share `out`, on rows of their own: it ends with the token of one of them,
    other callers draw theirs, and no slot stays taken."""
    import torch
    ident("sample_forward with a shared out")
    rng = np.random.default_rng(78)
    n = 151936
    rows = [rand_bf16(rng, n, 2.0) for _ in range(4)]
    xs = [dev(r) for r in rows]
    want = [oracle.sample(r, 0.8, 0.5) for r in rows]
    streams = [torch.cuda.Stream() for _ in rows]
    shared, own = (torch.zeros(k, dtype=torch.int32, device="cuda") for k in (1, 40))
    torch.cuda.synchronize()
    for i in range(40):
        for x, s in zip(xs[:3], streams):
            gpu.sample_forward(shared, x, n, 0.8, 0.5, stream=s)
        gpu.sample_forward(own[i:], xs[3], n, 0.8, 0.5, stream=streams[3])
    torch.cuda.synchronize()
    assert int(shared.item()) in want[:3]
    assert own.tolist() == [want[3]] * 40
    assert gpu.lib().llm_sample_slots(-1) == 0


def test_sample_forward_two_instances_of_a_graph(gpu, oracle):
    """One captured draw, instantiated twice and launched on two streams at once, with eager draws
    beside it: both instances have the same inputs and the same `out`, and give the same token."""
    import ctypes
    import torch
    from llm_inference_amd import model
    ident("sample_forward in two instances of a graph")
    rt = model._hip()
    rng = np.random.default_rng(79)
    n = 151936
    rows = [rand_bf16(rng, n, 2.0) for _ in range(2)]
    xs = [dev(r) for r in rows]
    want = [oracle.sample(r, 0.8, 0.5) for r in rows]
    out, eager = (torch.zeros(k, dtype=torch.int32, device="cuda") for k in (1, 30))
    streams = [torch.cuda.Stream() for _ in range(3)]
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    torch.cuda.synchronize()
    with torch.cuda.stream(streams[0]):
        graph.capture_begin()
        gpu.sample_forward(out, xs[0], n, 0.8, 0.5)
        graph.capture_end()
    execs = [ctypes.c_void_p() for _ in range(2)]
    raw = ctypes.c_void_p(graph.raw_cuda_graph())
    for e in execs:
        assert rt.hipGraphInstantiate(ctypes.byref(e), raw, None, None, ctypes.c_size_t(0)) == 0
    try:
        for i in range(30):
            out.fill_(-7)
            torch.cuda.synchronize()
            for _ in range(3):
                for e, s in zip(execs, streams):
                    assert rt.hipGraphLaunch(e, ctypes.c_void_p(s.cuda_stream)) == 0
            gpu.sample_forward(eager[i:], xs[1], n, 0.8, 0.5, stream=streams[2])
            torch.cuda.synchronize()
            assert int(out.item()) == want[0]
        assert eager.tolist() == [want[1]] * 30
        assert gpu.lib().llm_sample_slots(-1) == 0
    finally:
        torch.cuda.synchronize()
        for e in execs:
            rt.hipGraphExecDestroy(e)


# ---------------------------------------------------------------- argmax

def test_argmax(gpu, oracle):
    import torch
    ident("argmax")
    rng = np.random.default_rng(40)
    cases = [rand_bf16(rng, 151936) for _ in range(5)]
    cases.append(bf16_bits(np.full(151936, 2.5)))                     # all equal -> 0
    x = rand_bf16(rng, 151936); x[[7, 90000, 151935]] = bf16_bits(np.full(3, 50.0)); cases.append(x)
    x = rand_bf16(rng, 151936); x[151935] = bf16_bits(np.float32(60.0)).item(); cases.append(x)
    cases.append(bf16_bits(np.full(1000, -np.inf)))                   # all -inf -> 0
    x = rand_bf16(rng, 5000); x[::3] = 0x7FC0; cases.append(x)        # NaNs never taken
    cases.append(np.full(17, 0x7FC0, np.uint16))                      # all NaN -> INT_MAX
    cases.append(rand_bf16(rng, 1))
    cases.append(rand_bf16(rng, 13))
    out = dev_i32([-5])
    for x in cases:
        gpu.argmax_forward(out, dev(x), x.size)
        torch.cuda.synchronize()
        assert int(out.cpu()[0]) == oracle.argmax(x)
    # an unaligned view (falls back to 2-byte loads)
    x = rand_bf16(rng, 1001)
    xd = dev(x)
    gpu.argmax_forward(out, xd[1:], 1000)
    torch.cuda.synchronize()
    assert int(out.cpu()[0]) == oracle.argmax(x[1:])


# around a thread's last chunk and the longest row one workgroup takes (24576)
@pytest.mark.parametrize("n", [1, 7, 9, 8191, 8192, 8200, 24575, 24576, 24577, 32769])
def test_argmax_one_and_two_launches(gpu, oracle, n):
    import torch
    ident(f"argmax row of {n}")
    rng = np.random.default_rng(n)
    out = dev_i32([-5])
    ties, tail, nan = rand_bf16(rng, n), rand_bf16(rng, n), rand_bf16(rng, n)
    ties[rng.integers(0, n, 9)] = bf16_bits(np.float32(9.0))
    tail[n - 1] = bf16_bits(np.float32(9.0)).item()
    nan[n // 2:] = 0x7FC0
    lowest = np.full(n, 0xFF80, np.uint16)  # -inf, then NaN
    lowest[n // 3:] = 0xFFFF
    for row in (ties, tail, nan, lowest, np.full(n, 0x8000, np.uint16), np.full(n, 0x7FC0, np.uint16)):
        xd = dev(np.concatenate([row[:1], row]))
        for x in (dev(row), xd[1:]):
            gpu.argmax_forward(out, x, n)
            assert int(out.item()) == oracle.argmax(row)
