"""GPU tests of the matrix-core products behind prompts, the stateless forward and batched decoding, at the edges of their
tiles: rows, columns and reduction lengths just below, at and above a tile or a 32-deep stage, K cut into parts, one slice
and several, unaligned sizes.

Tolerances.  Split products: what is left out of a product of two f32 is below 2^-23 of it and the sums run over at most a
few thousand terms in f32, so 2e-5 of the largest value (the bound of the other many-token tests).  Projections: bit for bit."""
import re

import numpy as np
import pytest
import torch

from oracle import bdh_oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def bda():
    if not torch.cuda.is_available():
        pytest.fail("no HIP device: the GPU tests must run on the MI355X box")
    import burn_dragon_amd

    return burn_dragon_amd


def rel_err(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-30)


@pytest.mark.parametrize("B,h,T,N,d", [(1, 1, 8, 34, 64), (2, 3, 31, 130, 68), (1, 4, 33, 2080, 128), (3, 4, 65, 512, 256),
                                       (1, 2, 127, 4096, 260), (1, 1, 129, 62, 512), (5, 2, 16, 96, 192)])
@pytest.mark.parametrize("rotary", ["rope", "alibi"])
def test_many_token_step_at_tile_edges(bda, corc, B, h, T, N, d, rotary):
    from burn_dragon_amd.recurrent import recurrent_attention

    rng = np.random.default_rng(T + N)
    x = np.maximum(rng.standard_normal((B, h, T, N)) - 0.3, 0).astype(np.float32)
    v = rng.standard_normal((B, T, d)).astype(np.float32)
    rho = (0.1 * rng.standard_normal((B, h, N, d))).astype(np.float32)
    rot = {"rope": orc.ROPE, "alibi": orc.ALIBI}[rotary]
    freqs = corc.build_freqs(N, rotary=rot)
    slopes = corc.default_alibi_slopes(h) if rotary == "alibi" else None
    q = corc.rotate(x, freqs, rot, 17).astype(np.float64)
    # the token loop in float64
    out, state = np.zeros((B, h, T, d)), rho.astype(np.float64)
    decay = np.ones(h) if slopes is None else np.exp(-np.asarray(slopes, np.float32)).astype(np.float64)
    for t in range(T):
        out[:, :, t] = np.einsum("bhn,bhnd->bhd", q[:, :, t], state)
        state = (state + q[:, :, t, :, None] * v[:, None, t, None, :]) * decay[None, :, None, None]
    rho_t = torch.from_numpy(rho).to(DEV)
    ctx = bda.ffi.default_context(0)
    try:
        ctx.set_option("state_step.dense_chunks", 1)
        got = recurrent_attention(torch.from_numpy(x).to(DEV), torch.from_numpy(v).to(DEV), rho_t, torch.from_numpy(freqs).to(DEV),
                                  17, bda.RotaryEmbedding.parse(rotary))
    finally:
        ctx.set_option("state_step.dense_chunks", -1)
    assert rel_err(got.cpu().numpy(), out) < 2e-5
    assert rel_err(rho_t.cpu().numpy(), state) < 2e-5


@pytest.mark.parametrize("M,T,d,h,N", [(2, 1, 32, 1, 4), (15, 1, 64, 3, 68), (16, 16, 96, 2, 60), (17, 1, 256, 4, 1040), (33, 11, 128, 2, 9000),
                                       (63, 7, 512, 2, 132), (64, 1, 512, 3, 66), (65, 13, 192, 4, 8256), (129, 43, 160, 1, 260),
                                       (520, 130, 64, 8, 16384), (70, 5, 36, 2, 70)])
def test_relu_lowrank_rows_at_tile_edges(bda, corc, M, T, d, h, N):
    """Every tile height (16, 32, 64, 128 rows), rows and columns that end inside a tile, and the unaligned fallback give the
    bits of the k-sequential chain, with and without gate."""
    from burn_dragon_amd.kernel import relu_lowrank

    rng = np.random.default_rng(M + N)
    B = M // T
    inp = (rng.standard_normal((B, h, T, d)) * np.exp2(rng.integers(-20, 8, (B, h, T, d)))).astype(np.float32)
    weight = (rng.standard_normal((h, d, N)) * np.exp2(rng.integers(-30, 8, (h, d, N)))).astype(np.float32)
    gate = np.maximum(rng.standard_normal((B, h, T, N)), 0).astype(np.float32)
    ref = corc.relu_lowrank(inp, weight)
    args = (torch.from_numpy(inp).to(DEV), torch.from_numpy(weight).to(DEV), None, 0.0, bda.BlockPattern1d.dense(64))
    ctx = bda.ffi.default_context(0)
    try:
        ctx.set_option("relu_lowrank.row", 0)
        got = relu_lowrank.fused_forward(*args).cpu().numpy()
        gated = relu_lowrank.fused_forward(*args, gate=torch.from_numpy(gate).to(DEV)).cpu().numpy()
    finally:
        ctx.set_option("relu_lowrank.row", 1)
    assert np.array_equal(got, ref)
    assert np.array_equal(gated, gate * ref)


@pytest.mark.parametrize("T,V,d", [(86, 69, 128), (100, 300, 260), (128, 256, 192)])
def test_many_rows_through_the_second_stage_and_the_head(bda, T, V, d):
    """256 rows and more take a wavefront per row in the encoder's second stage and share the head's weights: the same rows in
    three smaller calls give the same logits to the rounding of the products before them (1e-5), the same greedy tokens."""
    cfg = bda.BDHConfig(n_layer=2, n_embd=d, n_head=2, mlp_internal_dim_multiplier=2, vocab_size=V)
    cfg.fused_kernels.set_rotary_embedding(bda.RotaryEmbedding.ALIBI)
    model = bda.BDH(cfg, DEV, seed=5)
    tokens = torch.randint(0, V, (3, T), generator=torch.Generator().manual_seed(T))
    logits, nxt = model.forward_with_state(tokens, model.init_state(), want_next=True)
    fast = model.forward_fast(tokens)
    for b in range(3):
        one, n1 = model.forward_with_state(tokens[b:b + 1], model.init_state(), want_next=True)
        assert rel_err(logits[b].cpu().numpy(), one[0].cpu().numpy()) < 1e-5
        assert rel_err(fast[b].cpu().numpy(), model.forward_fast(tokens[b:b + 1])[0].cpu().numpy()) < 1e-5
        assert int(nxt[b]) == int(n1[0]) == int(logits[b, -1].argmax())


@pytest.mark.parametrize("T", [9, 31, 33, 65, 520])
@pytest.mark.parametrize("slope", [4.0, 80.0, 120.0])
def test_steep_decay_over_a_ragged_prompt(bda, corc, T, slope):
    """A prompt that ends inside a 32-deep stage, through the dense form, with a state that loses up to e^-80 per
    token or, at a slope of 120 (whose factor rounds to zero), all of it."""
    from burn_dragon_amd.recurrent import recurrent_attention

    B, h, N, d = 2, 2, 96, 128
    rng = np.random.default_rng(T)
    x = np.maximum(rng.standard_normal((B, h, T, N)) - 0.3, 0).astype(np.float32)
    v = rng.standard_normal((B, T, d)).astype(np.float32)
    rho = (0.1 * rng.standard_normal((B, h, N, d))).astype(np.float32)
    slopes = np.array([slope, 0.5], np.float32)
    out, state = np.zeros((B, h, T, d)), rho.astype(np.float64)
    decay = np.exp(-slopes).astype(np.float64)
    for t in range(T):
        out[:, :, t] = np.einsum("bhn,bhnd->bhd", x[:, :, t].astype(np.float64), state)
        state = (state + x[:, :, t, :, None].astype(np.float64) * v[:, None, t, None, :]) * decay[None, :, None, None]
    rho_t = torch.from_numpy(rho).to(DEV)
    got = recurrent_attention(torch.from_numpy(x).to(DEV), torch.from_numpy(v).to(DEV), rho_t, torch.zeros(N, device=DEV), 0,
                              bda.RotaryEmbedding.ALIBI, slopes)
    for hh in range(h):
        assert rel_err(got.cpu().numpy()[:, hh], out[:, hh]) < 2e-5
        assert rel_err(rho_t.cpu().numpy()[:, hh], state[:, hh]) < 2e-5 or np.abs(state[:, hh]).max() < 1e-30


@pytest.mark.parametrize("M,d,N", [(8, 2050, 10), (63, 2052, 6), (9, 4100, 4), (8, 16388, 3), (40, 2080, 7)])
def test_relu_lowrank_wide_rows(bda, corc, M, d, N):
    """Eight rows and more of a width that neither comes in 16-byte pieces nor fits into LDS: the bits of the k-sequential
    chain."""
    from burn_dragon_amd.kernel import relu_lowrank

    h = 2
    rng = np.random.default_rng(M + N)
    inp = rng.standard_normal((M, h, 1, d)).astype(np.float32)
    weight = rng.standard_normal((h, d, N)).astype(np.float32)
    ref = corc.relu_lowrank(inp, weight)
    got = relu_lowrank.fused_forward(torch.from_numpy(inp).to(DEV), torch.from_numpy(weight).to(DEV), None, 0.0,
                                     bda.BlockPattern1d.dense(64))
    assert np.array_equal(got.cpu().numpy(), ref)


@pytest.mark.parametrize("kind,dtype,B,N,T,dense", [
    ("lazy", torch.float32, 3, 8192, 16, False), ("lazy", torch.float32, 3, 8192, 32, True),
    ("rope", torch.float32, 3, 8192, 24, False), ("rope", torch.float32, 3, 8192, 64, True),
    ("rope", torch.bfloat16, 16, 2048, 24, False), ("rope", torch.bfloat16, 16, 2048, 64, True),
    ("lazy", torch.bfloat16, 3, 8192, 16, False), ("lazy", torch.bfloat16, 3, 8192, 48, True)])
def test_short_prompts_walk_the_state_where_that_is_faster_at_five_percent(bda, kind, dtype, B, N, T, dense):
    """With 5 % of the neurons active the loop takes between 0.4 and 0.75 of the products' time in the cases marked False, and
    is the slower one in the others.  Which form ran shows in the bits: the loop's are those of state_step.dense_chunks = 0."""
    from burn_dragon_amd.kernel.linear_attention import build_freqs
    from burn_dragon_amd.recurrent import recurrent_attention, recurrent_attention_lazy_alibi

    h, d = 4, 256
    g = torch.Generator(device=DEV).manual_seed(T + N)
    x = torch.relu(torch.randn((B, h, T, N), device=DEV, generator=g) - 1.645)
    v = torch.randn((B, T, d), device=DEV, generator=g)
    rho = (0.01 * torch.randn((B, h, N, d), device=DEV, generator=g)).to(dtype)
    freqs = build_freqs(N, 65536.0, bda.RotaryEmbedding.ROPE, device=DEV).reshape(-1)
    ctx = bda.ffi.default_context(0)
    outs = []
    for mode in (0, -1):
        state = rho.clone()
        try:
            ctx.set_option("state_step.dense_chunks", mode)
            if kind == "rope":
                outs.append(recurrent_attention(x, v, state, freqs, 7, bda.RotaryEmbedding.ROPE))
            else:
                stamps = torch.full((B, h, N), 7, device=DEV, dtype=torch.int32)
                outs.append(recurrent_attention_lazy_alibi(x, v, state, stamps, 7))
        finally:
            ctx.set_option("state_step.dense_chunks", -1)
    assert torch.equal(outs[0], outs[1]) == (not dense)


@pytest.mark.parametrize("B,d,h,mult", [(48, 512, 8, 4), (24, 256, 4, 8), (33, 68, 2, 3), (64, 192, 4, 5), (65, 260, 2, 16),
                                        (300, 64, 2, 2), (40, 640, 2, 2), (26, 256, 4, 128)])
def test_batched_decode_encoder_on_the_matrix_cores(bda, B, d, h, mult):
    """The encoder E of a batch of decoding sequences: row tiles of 16, 32 and 64, rows and columns that end inside a tile, a
    reduction that is no multiple of a 32-deep stage, k-blocks added up in one workgroup and in the second stage.  The bits
    of the VALU kernel, except in the last case, which is large enough for the form with one chain per block of 1024: there
    and where that form is forced, 2^-24 per step of a few dozen steps, 1e-5."""
    cfg = bda.BDHConfig(n_layer=1, n_embd=d, n_head=h, mlp_internal_dim_multiplier=mult, vocab_size=64)
    cfg.fused_kernels.set_rotary_embedding(bda.RotaryEmbedding.ALIBI)
    model = bda.BDH(cfg, DEV, seed=3)
    N = mult * d // h
    g = torch.Generator(device=DEV).manual_seed(B)
    rho = 0.1 * torch.randn((1, B, h, N, d), device=DEV, generator=g)
    tokens = torch.randint(0, 64, (B, 1), device=DEV, generator=g)
    ctx = bda.ffi.default_context(0)
    logits = {}
    ctx.set_option("model.one_launch", 0)
    try:
        for rows in (24, -24, 1 << 30):
            ctx.set_option("decoder.splitk_rows", rows)
            state = model.init_state()
            state.position, state.storage = 9, rho.clone()
            state.layers[0].rho = state.storage[0]
            logits[rows] = model.forward_with_state(tokens, state).clone()
    finally:
        ctx.set_option("decoder.splitk_rows", 24)
        ctx.set_option("model.one_launch", 1)
    valu = logits[1 << 30]
    assert torch.equal(logits[24], valu) == (mult < 128)
    assert rel_err(logits[24].cpu().numpy(), valu.cpu().numpy()) < 1e-5
    assert rel_err(logits[-24].cpu().numpy(), valu.cpu().numpy()) < 1e-5


@pytest.mark.parametrize("B,T,d", [(8, 1, 516), (13, 1, 768), (3, 5, 640), (23, 1, 1024), (30, 1, 1024)])
def test_encoder_of_wide_rows_covers_every_row(bda, B, T, d):
    """Rows wider than 512, eight and more of them: each sequence gets the logits of a call of its own (other orders of the
    sums over 1024 and fewer terms: 1e-5)."""
    cfg = bda.BDHConfig(n_layer=2, n_embd=d, n_head=2, mlp_internal_dim_multiplier=1, vocab_size=64)
    cfg.fused_kernels.set_rotary_embedding(bda.RotaryEmbedding.ALIBI)
    model = bda.BDH(cfg, DEV, seed=3)
    tokens = torch.randint(0, 64, (B, T + 1), generator=torch.Generator().manual_seed(d))

    def last(rows):
        state = model.init_state()
        model.forward_with_state(tokens[rows, :1], state)  # the first token reads an empty state: nothing to encode
        return model.forward_with_state(tokens[rows, 1:], state).cpu().numpy()

    whole = last(slice(0, B))
    for b in range(B):
        assert rel_err(whole[b], last(slice(b, b + 1))[0]) < 1e-5


@pytest.mark.parametrize("T,N,d", [(128, 256, 256), (200, 256, 256), (2048, 256, 64)])
def test_split_products_round_the_large_sum_once(bda, T, N, d):
    """Row-normalised attention against float64.  A sum of K = 256 products is rounded K / 16 times on the way, the relative
    error of one rounding being at most 2^-24 and 2^-25.8 in the mean square, over sums that grow: sqrt(16 / 3) * 2^-25.8 =
    0.4e-7 for the scores, their own rounding, and as much again for the second product; 1.8e-7 = 3 * 2^-24 leaves room for a
    factor of two.  Sums rounded at each of the six instructions of a step are at 2.7e-7."""
    from burn_dragon_amd.kernel.linear_attention import build_freqs, default_alibi_slopes, fused_state_aligned

    h, block = 2, 64
    g = torch.Generator(device=DEV).manual_seed(T)
    q = torch.relu(torch.randn((1, h, T, N), device=DEV, generator=g))
    v = torch.randn((1, 1, T, d), device=DEV, generator=g)
    slopes = torch.tensor(default_alibi_slopes(h))
    out = fused_state_aligned(q, v, build_freqs(N, 65536.0, bda.RotaryEmbedding.ALIBI, device=DEV), slopes,
                              bda.BlockPattern2d.dense(block), bda.RotaryEmbedding.ALIBI)
    i = torch.arange(T, device=DEV)
    S = torch.matmul(q.double(), q.double().transpose(-1, -2).contiguous())
    S = torch.where(i[None, :] < i[:, None], S, 0.0)
    bias = slopes.to(DEV).double()[None, :, None, None] * (i[None, :] - i[:, None]).double()
    S = torch.where(i[None, :] // block <= i[:, None] // block, S + bias, 0.0)
    ref = torch.matmul(S, v.double().expand(1, h, T, d).contiguous()) / (S.abs().sum(-1, keepdim=True) + 1e-6)
    assert float((out.double() - ref).norm() / ref.norm()) < 1.8e-7


@pytest.mark.parametrize("M,d,h,N", [(7, 130, 2, 515), (16, 250, 4, 1022), (24, 256, 4, 515), (31, 384, 4, 1030), (31, 200, 3, 67),
                                     (32, 384, 4, 1030), (33, 100, 2, 9001), (63, 250, 4, 1022), (63, 700, 2, 30)])
def test_relu_lowrank_without_16_byte_pieces(bda, corc, M, d, h, N):
    """Widths that no 16-byte access fits, around the lines between the few-outputs kernel, the thread-per-column kernel and
    the checked matrix-core tiles: the bits of the k-sequential chain."""
    from burn_dragon_amd.kernel import relu_lowrank

    rng = np.random.default_rng(M + N)
    inp = rng.standard_normal((M, 1, 1, d)).astype(np.float32)
    weight = rng.standard_normal((h, d, N)).astype(np.float32)
    got = relu_lowrank.fused_forward(torch.from_numpy(inp).to(DEV), torch.from_numpy(weight).to(DEV), None, 0.0,
                                     bda.BlockPattern1d.dense(64))
    assert np.array_equal(got.cpu().numpy(), corc.relu_lowrank(inp, weight))


@pytest.mark.parametrize("rows,d", [(3, 4096), (512, 36), (513, 36), (515, 1001), (2, 4100), (600, 4097)])
def test_layer_norm_one_and_four_rows_per_workgroup(bda, corc, rows, d):
    from burn_dragon_amd.recurrent import layer_norm

    x = np.random.default_rng(d).standard_normal((rows, d)).astype(np.float32)
    assert np.array_equal(layer_norm(torch.from_numpy(x).to(DEV)).cpu().numpy(), corc.layer_norm(x))


@pytest.mark.parametrize("kind", ["rope", "lazy"])
def test_prompt_without_room_for_the_dense_form_is_walked(bda, kind):
    """A bf16 state whose f32 copy does not fit: the token loop's bits, no error; an error where the dense form was asked for."""
    from burn_dragon_amd.kernel.linear_attention import build_freqs
    from burn_dragon_amd.recurrent import recurrent_attention, recurrent_attention_lazy_alibi

    B, h, T, N, d = 4, 4, 96, 8192, 256  # 128 MiB of f32 state
    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.relu(torch.randn((B, h, T, N), device=DEV, generator=g) - 1.645)
    v = torch.randn((B, T, d), device=DEV, generator=g)
    rho = (0.01 * torch.randn((B, h, N, d), device=DEV, generator=g)).bfloat16()
    stamps = torch.randint(0, 8, (B, h, N), device=DEV, generator=g, dtype=torch.int32)
    freqs = build_freqs(N, 65536.0, bda.RotaryEmbedding.ROPE, device=DEV).reshape(-1)

    def call(mib, mode):
        ctx = bda.ffi.Context(0)
        ctx.set_option("workspace.max_mib", mib)
        ctx.set_option("state_step.dense_chunks", mode)
        state, at = rho.clone(), stamps.clone()
        if kind == "rope":
            out = recurrent_attention(x, v, state, freqs, 7, bda.RotaryEmbedding.ROPE, ctx=ctx)
        else:
            out = recurrent_attention_lazy_alibi(x, v, state, at, 7, ctx=ctx)
        torch.cuda.synchronize()
        return out, state, at

    walked, short, dense = call(0, 0), call(72, -1), call(0, -1)
    assert all(torch.equal(a, b) for a, b in zip(walked, short))
    assert not torch.equal(dense[0], walked[0])  # with room the products are taken
    with pytest.raises(bda.ffi.BdhError):
        call(72, 1)


@pytest.mark.parametrize("d,h,N,B,T", [
    (128, 2, 66, 3, 45),    # rows of several sequences in one tile, columns that end inside it
    (256, 4, 1024, 2, 64),  # whole tiles
    (36, 1, 131, 1, 100),   # a k that ends inside a stage, odd rows of the weights
    (512, 2, 96, 1, 130),
    (256, 4, 8192, 1, 200),  # by size
])
def test_gated_projection_of_a_prompt_on_split_products(d, h, N, B, T):
    """D_y of a prompt and of the stateless form as split-bf16 products against the f32 chain: sums of d terms in another
    order, 2^-24 a step, through two layers and a few thousand terms of the encoder: 1e-5."""
    import burn_dragon_amd as bda

    cfg = bda.BDHConfig(n_layer=2, n_embd=d, n_head=h, mlp_internal_dim_multiplier=1, vocab_size=64, dropout=0.0)
    cfg.latent_per_head = lambda: N
    cfg.fused_kernels.set_rotary_embedding(bda.RotaryEmbedding.ALIBI)
    model = bda.BDH(cfg, DEV, seed=3)
    g = torch.Generator(device=DEV).manual_seed(N)
    tokens = torch.randint(0, 64, (B, T), device=DEV, generator=g)
    ctx = bda.ffi.default_context(0)
    got = []
    for split in (0, -1 if N == 8192 else 1):
        ctx.set_option("relu_lowrank.split", split)
        try:
            state = model.init_state()
            logits = model.forward_with_state(tokens, state)
            got.append((logits, model.forward_fast(tokens), state.storage))
            torch.cuda.synchronize()
        finally:
            ctx.set_option("relu_lowrank.split", -1)
    for a, b in zip(*got):
        assert not torch.equal(a, b)
        assert float((a - b).abs().max() / a.abs().max()) < 1e-5


@pytest.mark.parametrize("d,h,N,B,T,tile", [
    (36, 1, 131, 1, 100, "k_gemm_f32_small<"), (128, 2, 66, 3, 45, "k_gemm_f32_small<"),
    (128, 2, 8192, 1, 100, "k_gemm_f32<64, 64"), (256, 4, 8192, 1, 200, "k_gemm_f32<128, 128"),
    (768, 4, 8192, 1, 200, "k_gemm_f32<128, 256"),
])
@pytest.mark.parametrize("where,value", [("weight", float("nan")), ("weight", float("inf")), ("weight", -float("inf")),
                                         ("weight", 3.4e38), ("weight", -3.4e38), ("weights", float("nan")),
                                         ("embedding", float("nan")), ("embedding", float("inf"))])
def test_gated_projection_of_numbers_that_no_split_holds(bda, d, h, N, B, T, tile, where, value):
    """D_y of a prompt and of the stateless form with weights and inputs that are infinite, NaN or beyond the largest bf16: on
    split products as in the f32 chain, where a NaN is not above the threshold and a finite weight keeps its value (what is a
    number to the bound of the test above, in the same places)."""
    cfg = bda.BDHConfig(n_layer=1, n_embd=d, n_head=h, mlp_internal_dim_multiplier=1, vocab_size=64, dropout=0.0)
    cfg.latent_per_head = lambda: N
    cfg.fused_kernels.set_rotary_embedding(bda.RotaryEmbedding.ROPE if N % 2 == 0 else bda.RotaryEmbedding.ALIBI)
    g = torch.Generator(device=DEV).manual_seed(N)
    normal = lambda *shape: 0.02 * torch.randn(shape, device=DEV, generator=g)
    weights = {"embed": 50 * normal(64, d), "encoder": normal(h, d, N), "encoder_v": normal(h, d, N), "decoder": normal(h * N, d),
               "lm_head": normal(d, 64)}
    if where == "embedding":
        weights["embed"][7, 3] = value
    else:
        weights["encoder_v"][0, 5, N - 2] = value
        if where == "weights":
            weights["encoder_v"][:, :, ::3] = value
    model = bda.BDH(cfg, DEV, weights=weights)
    tokens = torch.randint(8, 64, (B, T), device=DEV, generator=g)
    tokens[0, T // 2] = 7
    ctx = bda.ffi.default_context(0)
    got = []
    for split in (0, 1):
        ctx.set_option("relu_lowrank.split", split)
        try:
            state = model.init_state()
            logits, ran = _launched(lambda: model.forward_with_state(tokens, state))
            got.append((logits, model.forward_fast(tokens), state.storage))
        finally:
            ctx.set_option("relu_lowrank.split", -1)
        assert (re.search(tile + r"[^>]*\b3>", ran) is not None) == (split == 1), ran  # 3: the gated epilogue
    for a, b in zip(*got):
        assert torch.equal(torch.isfinite(a), torch.isfinite(b))
        a, b = (torch.where(torch.isfinite(t), t, 0.0) for t in (a, b))
        assert float((a - b).abs().max()) <= 1e-5 * float(a.abs().max())
    assert bool(torch.isfinite(got[0][0][:, : T // 2]).all(-1).any())


def _launched(call):
    from torch.profiler import ProfilerActivity, profile

    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        out = call()
        torch.cuda.synchronize()
    return out, " ".join(e.key for e in prof.key_averages())


@pytest.mark.parametrize("d,h,N,T,split", [
    (128, 4, 12288, 1, False), (128, 4, 12288, 32, False), (128, 4, 12288, 33, True),    # few rows: the weights bound them
    (256, 4, 16384, 16, False), (256, 4, 16384, 17, True), (260, 4, 12289, 8, False), (260, 4, 12289, 9, True),
    (128, 4, 12288, 129, False), (128, 4, 12288, 193, True), (128, 4, 8192, 129, True),  # padding to whole tiles
    (192, 4, 6144, 257, False), (192, 4, 6144, 385, True), (192, 4, 12288, 257, True),
])
def test_where_the_gated_projection_takes_split_products(bda, d, h, N, T, split):
    """The rows from which on split products are faster than the f32 chain."""
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("rounds of 256 CUs")
    cfg = bda.BDHConfig(n_layer=1, n_embd=d, n_head=h, mlp_internal_dim_multiplier=1, vocab_size=64)
    cfg.latent_per_head = lambda: N
    cfg.fused_kernels.set_rotary_embedding(bda.RotaryEmbedding.ALIBI)
    model = bda.BDH(cfg, DEV, seed=3)
    _, ran = _launched(lambda: model.forward_fast(torch.zeros((1, T), device=DEV, dtype=torch.int64)))
    assert (re.search(r"k_gemm_f32(_small)?<[^>]*\b3>", ran) is not None) == split, ran


@pytest.mark.parametrize("rotary", ["rope", "alibi", "pope"])
@pytest.mark.parametrize("B,h,T,N,d", [
    (1, 2, 8, 16, 32),     # one step of k for one of the four wavefronts, tiles that end inside
    (1, 3, 33, 62, 36),    # a k that ends inside a step, in every product; a second row tile of one row
    (2, 2, 65, 34, 100),   # rows that are no whole 16-byte pieces
    (1, 4, 128, 256, 256),
    (1, 1, 200, 250, 64),
])
def test_products_of_few_tiles(bda, rotary, B, h, T, N, d):
    """32 x 32 tiles whose wavefronts share K: scores, readout and state of a short prompt against the loop over its tokens, the
    same sums reassociated (a few hundred terms, 2^-24 each): 2e-5 as for the other tiles; the stateless form (time blocks,
    additive ALiBi terms, row norms) against itself in float64."""
    from burn_dragon_amd.recurrent import recurrent_attention

    g = torch.Generator(device=DEV).manual_seed(T + N)
    rot = bda.RotaryEmbedding.parse(rotary)
    x = torch.relu(torch.randn((B, h, T, N), device=DEV, generator=g))
    v = torch.randn((B, T, d), device=DEV, generator=g)
    rho = 0.1 * torch.randn((B, h, 2 * N if rotary == "pope" else N, d), device=DEV, generator=g)
    freqs = torch.rand(N, device=DEV, generator=g).repeat_interleave(2)[:N].contiguous()
    ctx = bda.ffi.default_context(0)
    got = []
    for mode in (0, 1):
        state = rho.clone()
        ctx.set_option("state_step.dense_chunks", mode)
        try:
            out, ran = _launched(lambda: recurrent_attention(x, v, state, freqs, 5, rot))
        finally:
            ctx.set_option("state_step.dense_chunks", -1)
        assert ("k_gemm_f32_small" in ran) == (mode == 1)
        got.append((out, state))
    for a, b in zip(*got):
        assert float((a - b).abs().max() / a.abs().max()) < 2e-5


@pytest.mark.parametrize("B,T,small", [(4, 200, False), (1, 256, True)])
def test_encoder_tiles_of_a_prompt_count_their_last_round(bda, B, T, small):
    """The encoder of 800 rows and 4 heads of 1024 neurons: 32 x 32 tiles would be 3.1 rounds of workgroups, and slower than 64 x
    64 tiles in parts; of 256 rows, one round, they are the faster ones."""
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("rounds of 256 CUs")
    cfg = bda.BDHConfig(n_layer=1, n_embd=256, n_head=4, mlp_internal_dim_multiplier=16, vocab_size=64)
    cfg.fused_kernels.set_rotary_embedding(bda.RotaryEmbedding.ROPE)
    model = bda.BDH(cfg, DEV, seed=3)
    tokens = torch.randint(0, 64, (B, T), generator=torch.Generator().manual_seed(T))
    _, ran = _launched(lambda: model.forward_with_state(tokens, model.init_state()))
    assert ("k_gemm_f32_small" in ran) == small


@pytest.mark.parametrize("T,N,d,block", [(130, 48, 36, 1), (129, 20, 32, 64), (160, 64, 64, 32)])
def test_row_norms_of_few_tiles(bda, T, N, d, block):
    """The stateless form on 32 x 32 tiles against its formula in float64: sums of up to 160 terms over their norm, 1e-5."""
    from burn_dragon_amd.kernel.block_sparse import BlockPattern2d
    from burn_dragon_amd.kernel.linear_attention import fused_state_aligned

    B, h = 2, 2
    g = torch.Generator(device=DEV).manual_seed(T)
    q = torch.relu(torch.randn((B, h, T, N), device=DEV, generator=g))
    v = torch.randn((B, 1, T, d), device=DEV, generator=g)
    slopes = torch.tensor([0.5, 0.25])
    freqs = torch.zeros((1, 1, 1, N), device=DEV)
    (out, ran) = _launched(lambda: fused_state_aligned(q, v, freqs, slopes, BlockPattern2d.dense(block), bda.RotaryEmbedding.ALIBI))
    assert "k_gemm_f32_small" in ran
    t = torch.arange(T, device=DEV)
    s = torch.matmul(q.double(), q.double().transpose(-1, -2).contiguous())
    same = t[:, None] // block == t[None] // block
    s = torch.where(same & (t[None] >= t[:, None]), torch.zeros_like(s), s)
    s = s + slopes.to(DEV).double()[:, None, None] * (t[None] - t[:, None]).double()
    s = torch.where(t[None] // block <= t[:, None] // block, s, torch.zeros_like(s))
    ref = torch.matmul(s, v.double()) / (s.abs().sum(-1, keepdim=True) + 1e-6)
    assert float((out.double() - ref).abs().max() / ref.abs().max()) < 1e-5
