"""The 128 x 256 tile of the split-bf16 products (two stages in LDS, two wavefronts of a SIMD in turns), which only large calls
take: row and column edges inside a tile, a reduction that ends inside a stage, operands that do not come in aligned pieces,
a second pair of operands, parts of K; and the state update's read-modify-write at ragged sizes."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("rotary,T,N,d", [("rope", 490, 4096, 256), ("rope", 491, 4098, 500), ("alibi", 490, 4096, 500),
                                          ("alibi", 487, 4097, 509), ("alibi", 130, 8192, 256)])
def test_wide_tile_against_float64(rotary, T, N, d):
    """out = tril(-1)(Q Q^T) V + Q rho, rho += Q^T V (ALiBi: with powers of the decay), frequencies of zero so that Q = x.
    Sums of up to 8192 terms rounded once per 16: 2^-24 * sqrt(512) = 1.4e-6 of a sum of equal terms; 4e-6 of the largest."""
    import burn_dragon_amd as bda
    from burn_dragon_amd.recurrent import recurrent_attention

    B, h = 3, 4
    rot = bda.RotaryEmbedding.parse(rotary)
    g = torch.Generator(device=DEV).manual_seed(T + N)
    x = torch.relu(torch.randn((B, h, T, N), device=DEV, generator=g))
    v = torch.randn((B, T, d), device=DEV, generator=g)
    rho = 0.1 * torch.randn((B, h, N, d), device=DEV, generator=g)
    before = rho.clone()
    freqs = torch.zeros(N, device=DEV)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        out = recurrent_attention(x, v, rho, freqs, 0, rot)
        torch.cuda.synchronize()
    names = [e.key for e in prof.key_averages()]
    assert any("k_gemm_f32<128, 256" in n for n in names), names
    decay = torch.ones(h, dtype=torch.float64, device=DEV)
    if rotary == "alibi":
        from burn_dragon_amd.kernel.linear_attention import default_alibi_slopes

        slopes = torch.as_tensor(default_alibi_slopes(h), dtype=torch.float32)
        decay = torch.exp(-slopes).double().to(DEV)
    t = torch.arange(T, device=DEV, dtype=torch.float64)
    for b in range(B):
        for i in range(h):
            q, val, r0 = x[b, i].double(), v[b].double(), before[b, i].double()
            powers = decay[i] ** (t[:, None] - t[None, :]).clamp_min(0)
            want = ((q @ q.T).tril(-1) * powers) @ val + (decay[i] ** t)[:, None] * (q @ r0)
            state = decay[i] ** T * r0 + ((decay[i] ** (T - t))[:, None] * q).T @ val
            assert float((out[b, i].double() - want).abs().max() / want.abs().max()) < 4e-6
            assert float((rho[b, i].double() - state).abs().max() / state.abs().max()) < 4e-6


@pytest.mark.parametrize("T,d", [(128, 256), (90, 260), (100, 512), (88, 516), (86, 1024)])
def test_rows_of_every_width_through_layer_norm_and_second_stage(T, d):
    """A wavefront holds a row in 4, 8 or 16 registers a lane once a call has 256 rows; a step has its own kernels.  Five stages,
    each a sum of up to 1024 terms: 5 * 2^-24 * sqrt(1024) = 1e-5 of the largest logit, twice that allowed."""
    import burn_dragon_amd as bda

    cfg = bda.BDHConfig(n_layer=1, n_embd=d, n_head=2, mlp_internal_dim_multiplier=1, vocab_size=40)
    cfg.fused_kernels.set_rotary_embedding(bda.RotaryEmbedding.ALIBI)
    model = bda.BDH(cfg, DEV, seed=d)
    tokens = torch.randint(0, 40, (3, T), generator=torch.Generator().manual_seed(T))
    logits = model.forward_with_state(tokens, model.init_state())
    state = model.init_state()
    for t in range(T):
        one = model.forward_with_state(tokens[:, t:t + 1], state)[:, 0]
        assert (logits[:, t] - one).abs().max() <= 2e-5 * one.abs().max()


@pytest.mark.parametrize("h,T,d,block", [(11, 511, 256, 1), (16, 450, 260, 64), (13, 500, 200, 48), (33, 321, 96, 1)])
def test_row_normalised_attention_in_small_tiles(h, T, d, block):
    """Chips full of 64 x 64 tiles: odd and even slices walk their row tiles in opposite orders, a time block crosses tiles or
    not.  Errors of a sum rounded once per 16 products, K = 64 and then T: sqrt(T / 48) * 2^-25.8 < 0.6e-7 for the second
    product, 0.4e-7 for the scores and as much for storing them; 3 * 2^-24 = 1.8e-7."""
    import burn_dragon_amd as bda
    from burn_dragon_amd.kernel.linear_attention import build_freqs, default_alibi_slopes, fused_state_aligned

    B, N = 3, 64
    g = torch.Generator(device=DEV).manual_seed(T)
    q = torch.relu(torch.randn((B, h, T, N), device=DEV, generator=g))
    v = torch.randn((B, 1, T, d), device=DEV, generator=g)
    slopes = torch.tensor(default_alibi_slopes(h))
    out = fused_state_aligned(q, v, build_freqs(N, 65536.0, bda.RotaryEmbedding.ALIBI, device=DEV), slopes,
                              bda.BlockPattern2d.dense(block), bda.RotaryEmbedding.ALIBI)
    i = torch.arange(T, device=DEV)
    S = torch.matmul(q.double(), q.double().transpose(-1, -2).contiguous())
    S = torch.where(i[None, :] < i[:, None], S, 0.0)
    bias = slopes.to(DEV).double()[None, :, None, None] * (i[None, :] - i[:, None]).double()
    S = torch.where(i[None, :] // block <= i[:, None] // block, S + bias, 0.0)
    ref = torch.matmul(S, v.double().expand(B, h, T, d).contiguous()) / (S.abs().sum(-1, keepdim=True) + 1e-6)
    for s in range(h):  # every slice: one in the wrong order would be wrong alone
        assert float((out[:, s].double() - ref[:, s]).norm() / ref[:, s].norm()) < 1.8e-7


@pytest.mark.parametrize("fresh", [False, True])
def test_prefill_of_rows_of_more_than_four_gib_a_tile(fresh):
    """34 M neurons, of which only the first and last few have activations: the bits of the call over those alone (every sum
    runs over k in order, and a zero adds nothing), the other rows of the state as they were."""
    from burn_dragon_amd.recurrent import prefill_chunked

    T, N, d, few = 64, 34_209_792, 8, 1024
    g = torch.Generator(device=DEV).manual_seed(3)
    x = torch.zeros((1, 1, T, N), device=DEV, dtype=torch.bfloat16)
    for part in (slice(0, few), slice(N - few, N)):
        x[..., part] = torch.relu(torch.randn((1, 1, T, few), device=DEV, generator=g)).bfloat16()
    v = torch.randn((1, T, d), device=DEV, generator=g).bfloat16()
    rho = torch.zeros((1, 1, N, d), device=DEV) if fresh else 0.1 * torch.randn((1, 1, N, d), device=DEV, generator=g)
    freqs = torch.rand(N, device=DEV, generator=g)

    def ends(t, dim):
        return torch.cat([t.narrow(dim, 0, few), t.narrow(dim, N - few, few)], dim).contiguous()

    x_few, rho_few, freqs_few, between = ends(x, 3), ends(rho, 2), ends(freqs, 0), rho[:, :, few:N - few].clone()
    out = prefill_chunked(x, v, rho, freqs, 5, state_is_zero=fresh)
    out_few = prefill_chunked(x_few, v, rho_few, freqs_few, 5, state_is_zero=fresh)
    assert torch.equal(out, out_few) and bool((out != 0).any())
    assert torch.equal(ends(rho, 2), rho_few)
    assert torch.equal(rho[:, :, few:N - few], between)
