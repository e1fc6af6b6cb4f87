"""The kernels of a decode step at the sizes where they can go wrong.  The two-launch layer: row widths at the edges of the
three kernel widths (128, 256, 512), one and many blocks of neurons, the smallest and largest number of them, blocks of 32
and of 64, vocabularies read four columns at a time and one at a time, weights that are not 16-byte aligned.  The projections
and the encoder of a few rows: rings of copies that are longer than the work, and tiles that end inside."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def rel_err(a, b):
    a, b = a.double().cpu(), b.double().cpu()
    return float((a - b).abs().max() / b.abs().max().clamp_min(1e-30))


@pytest.mark.parametrize("state", ["f32", "bf16"])
@pytest.mark.parametrize("rotary,lazy", [("rope", False), ("pope", False), ("alibi", False), ("alibi", True)])
@pytest.mark.parametrize("d,h,N,V,B,aligned", [
    (128, 1, 64, 69, 1, True),      # two blocks of 32
    (128, 4, 128, 1024, 17, True),  # sixteen blocks of 32 a sequence, more workgroups than a chip of 256 has
    (132, 3, 64, 1021, 2, True),    # a row that barely leaves the narrowest kernel
    (252, 3, 192, 40, 3, True),     # rows that do not fill the middle kernel, blocks no multiple of its access
    (256, 2, 1024, 256, 2, True),   # 64 blocks of 32
    (256, 4, 1024, 64, 2, True),    # 64 blocks of 64
    (260, 1, 64, 516, 1, True),
    (512, 4, 64, 1024, 3, True),
    (128, 4, 32, 69, 3, True),      # a single block of 32 per head
    (192, 4, 96, 256, 40, True),    # an odd number of them, more workgroups than a chip of 256 has at once
    (512, 2, 1024, 64, 1, True),    # 64 blocks of 32
    (128, 1, 2016, 33, 2, True),    # 63 blocks of 32
    (256, 4, 128, 256, 2, False),   # weights four bytes off
    (128, 1, 128, 64, 400, True),   # more sequences than a chip of 256 takes in one round of the one-launch step
])
def test_two_launch_layer_edges(state, rotary, lazy, d, h, N, V, B, aligned):
    import burn_dragon_amd as bda
    from burn_dragon_amd import ffi

    cfg = bda.BDHConfig(n_layer=2, n_embd=d, n_head=h, mlp_internal_dim_multiplier=1, vocab_size=V, dropout=0.0)
    # N per head is multiplier * n_embd / n_head: choose the neurons directly
    cfg.latent_per_head = lambda: N
    cfg.fused_kernels.set_rotary_embedding(bda.RotaryEmbedding.parse(rotary))
    g = torch.Generator(device=DEV).manual_seed(d + N)
    w = {"embed": torch.randn((V, d), device=DEV, generator=g)}
    for name, shape in (("encoder", (h, d, N)), ("encoder_v", (h, d, N)), ("decoder", (h * N, d)), ("lm_head", (d, V))):
        w[name] = 0.05 * torch.randn(shape, device=DEV, generator=g)
    if not aligned:  # four bytes off
        for name, t in w.items():
            flat = torch.empty(t.numel() + 1, device=DEV)
            flat[1:] = t.reshape(-1)
            w[name] = flat[1:].view(t.shape)
    models = [bda.BDH(cfg, DEV, weights=w, alibi_lazy=lazy, rho_dtype=ffi.BF16 if state == "bf16" else ffi.F32) for _ in range(2)]
    assert all((t.data_ptr() % 16 == 0) == aligned for t in models[0].params.values())
    ctx = bda.ffi.default_context(0)
    states = [m.init_state() for m in models]
    start = 0.1 * torch.randn((2, B, h, models[0].latent_q, d), device=DEV, generator=g)
    for m, s in zip(models, states):
        m._ensure_state(s, B)
        s.storage.copy_(start)
        s.position = 5
        if lazy:
            s.stamps.fill_(3)  # two tokens of decay pending
    tokens = torch.randint(0, V, (3, B, 1), device=DEV, generator=g)
    assert all(k in _kernels_of_a_step(models[0], B) for k in ("k_layer_phase_a", "k_layer_phase_b"))
    for t in range(3):
        got, nxt = models[0].forward_with_state(tokens[t], states[0], want_next=True)
        try:
            ctx.set_option("model.one_launch", 0)
            ref = models[1].forward_with_state(tokens[t], states[1])
        finally:
            ctx.set_option("model.one_launch", 1)
        torch.cuda.synchronize()
        # f32: other summation trees over at most 4096 terms.  bf16: the inputs of a rounding differ in their last bits, so a
        # stored element may land one bf16 step (2^-8 of it) apart; thousands of them average out in a readout
        assert rel_err(got, ref) < (1e-5 if state == "f32" else 2e-3), t
        assert torch.equal(nxt.reshape(-1), got[:, 0].argmax(-1))
    for m, s in zip(models, states):
        m.materialize_state(s)
    torch.cuda.synchronize()
    assert rel_err(states[0].storage.float(), states[1].storage.float()) < (1e-5 if state == "f32" else 3 * 2.0 ** -8)
    if lazy:
        assert torch.equal(states[0].stamps, states[1].stamps)


@pytest.mark.parametrize("d,h,N,V,B,aligned", [
    (128, 4, 128, 64, 1, True),    # one block of 64 columns
    (128, 4, 128, 69, 3, True),    # ... and one that starts within it
    (132, 4, 64, 127, 2, True),
    (256, 4, 128, 128, 2, True),
    (256, 2, 1024, 1021, 2, False),  # 64 partial rows, weights four bytes off
    (512, 4, 64, 1024, 3, True),
    (256, 4, 128, 63, 1, True),    # too few columns: one workgroup
])
def test_logits_without_a_greedy_token(d, h, N, V, B, aligned):
    """The logits of a step that wants no token, 64 columns a workgroup, against those of one that does: sums of at most 512
    terms in another order, 1e-5."""
    import burn_dragon_amd as bda

    cfg = bda.BDHConfig(n_layer=2, n_embd=d, n_head=h, mlp_internal_dim_multiplier=1, vocab_size=V, dropout=0.0)
    cfg.latent_per_head = lambda: N
    g = torch.Generator(device=DEV).manual_seed(d + V)
    w = {"embed": torch.randn((V, d), device=DEV, generator=g)}
    for name, shape in (("encoder", (h, d, N)), ("encoder_v", (h, d, N)), ("decoder", (h * N, d)), ("lm_head", (d, V))):
        w[name] = 0.05 * torch.randn(shape, device=DEV, generator=g)
    if not aligned:
        flat = torch.empty(d * V + 1, device=DEV)
        flat[1:] = w["lm_head"].reshape(-1)
        w["lm_head"] = flat[1:].view(d, V)
    models = [bda.BDH(cfg, DEV, weights=w) for _ in range(2)]
    states = [m.init_state() for m in models]
    assert ("k_phase_logits" in _kernels_of_a_step(models[0], B)) == (V >= 64)
    tokens = torch.randint(0, V, (2, B, 1), device=DEV, generator=g)
    for t in range(2):
        got = models[0].forward_with_state(tokens[t], states[0])
        ref, _ = models[1].forward_with_state(tokens[t], states[1], want_next=True)
        torch.cuda.synchronize()
        assert rel_err(got, ref) < 1e-5, t


@pytest.mark.parametrize("d", [128, 200, 512])
@pytest.mark.parametrize("V", [2, 3, 4, 61, 64, 65, 128, 129, 257])
def test_greedy_head_of_few_and_ragged_columns(d, V):
    """One column and four at a time, the last four of a row overlapping; spans of k added within a wave (up to 64 and 128
    columns) and across waves: against the kernel-by-kernel step, sums of at most 512 terms in another order, 1e-5."""
    import burn_dragon_amd as bda

    cfg = bda.BDHConfig(n_layer=1, n_embd=d, n_head=2, mlp_internal_dim_multiplier=1, vocab_size=V, dropout=0.0)
    cfg.latent_per_head = lambda: 64
    g = torch.Generator(device=DEV).manual_seed(d + V)
    w = {"embed": torch.randn((V, d), device=DEV, generator=g)}
    for name, shape in (("encoder", (2, d, 64)), ("encoder_v", (2, d, 64)), ("decoder", (128, d)), ("lm_head", (d, V))):
        w[name] = 0.05 * torch.randn(shape, device=DEV, generator=g)
    models = [bda.BDH(cfg, DEV, weights=w) for _ in range(2)]
    states = [m.init_state() for m in models]
    ctx = bda.ffi.default_context(0)
    tokens = torch.randint(0, V, (2, 3, 1), device=DEV, generator=g)
    for t in range(2):
        got, nxt = models[0].forward_with_state(tokens[t], states[0], want_next=True)
        try:
            ctx.set_option("model.one_launch", 0)
            ref = models[1].forward_with_state(tokens[t], states[1])
        finally:
            ctx.set_option("model.one_launch", 1)
        torch.cuda.synchronize()
        assert rel_err(got, ref) < 1e-5, t
        assert torch.equal(nxt.reshape(-1), got[:, 0].argmax(-1))


@pytest.mark.parametrize("d,h,N,aligned", [
    (256, 4, 8192, True),   # 128 columns a workgroup, one for every CU of a chip of 256
    (256, 4, 8190, True),   # ... the last one not full, rows that are no whole 16-byte pieces
    (256, 4, 4100, True),   # 64 columns a workgroup, the last one with four
    (256, 4, 8192, False),  # weights four bytes off
    (512, 1, 70, True),     # 32 columns a workgroup, one partial row
    (512, 2, 4092, True),
    (512, 1, 4092, False),
])
def test_projections_of_one_row_that_make_their_row(d, h, N, aligned):
    """The four-launch layer at the edges of its projections' workgroups, against the kernel-by-kernel step: sums of at most
    512 terms in another order, 1e-5."""
    import burn_dragon_amd as bda

    V = 64
    cfg = bda.BDHConfig(n_layer=2, n_embd=d, n_head=h, mlp_internal_dim_multiplier=1, vocab_size=V, dropout=0.0)
    cfg.latent_per_head = lambda: N
    cfg.fused_kernels.set_rotary_embedding(bda.RotaryEmbedding.ROPE)
    g = torch.Generator(device=DEV).manual_seed(d + N)
    w = {"embed": torch.randn((V, d), device=DEV, generator=g)}
    for name, shape in (("encoder", (h, d, N)), ("encoder_v", (h, d, N)), ("decoder", (h * N, d)), ("lm_head", (d, V))):
        w[name] = 0.05 * torch.randn(shape, device=DEV, generator=g)
    if not aligned:  # four bytes off
        for name, t in w.items():
            flat = torch.empty(t.numel() + 1, device=DEV)
            flat[1:] = t.reshape(-1)
            w[name] = flat[1:].view(t.shape)
    models = [bda.BDH(cfg, DEV, weights=w) for _ in range(2)]
    assert all((t.data_ptr() % 16 == 0) == aligned for t in models[0].params.values())
    ctx = bda.ffi.default_context(0)
    states = [m.init_state() for m in models]
    start = 0.1 * torch.randn((2, 1, h, N, d), device=DEV, generator=g)
    for m, s in zip(models, states):
        m._ensure_state(s, 1)
        s.storage.copy_(start)
        s.position = 5
    tokens = torch.randint(0, V, (3, 1, 1), device=DEV, generator=g)
    assert "k_relu_lowrank_row1" in _kernels_of_a_step(models[0], 1)
    for t in range(3):
        got, nxt = models[0].forward_with_state(tokens[t], states[0], want_next=True)
        try:
            ctx.set_option("model.fused_rows", 0)
            ref = models[1].forward_with_state(tokens[t], states[1])
        finally:
            ctx.set_option("model.fused_rows", 1)
        torch.cuda.synchronize()
        assert rel_err(got, ref) < 1e-5, t
        assert torch.equal(nxt.reshape(-1), got[:, 0].argmax(-1))
    assert rel_err(states[0].storage, states[1].storage) < 1e-5


@pytest.mark.parametrize("d", [32, 64, 96, 160, 256, 512])
@pytest.mark.parametrize("B,T,h,N", [(2, 1, 3, 4), (5, 3, 2, 60), (17, 1, 3, 68), (33, 1, 1, 260), (63, 1, 2, 64),
                                     (20, 1, 2, 40960), (40, 1, 1, 66000)])
def test_projection_rings_keep_the_bits_of_the_scalar_chain(d, B, T, h, N):
    """1 to 16 stages of 32 k through rings of 2, 3 and 4 and, where there are few workgroups, all of them at once; row tiles of 16, 32 and 64; bias, mask and gate: the bits of the
    thread-per-column kernel, which adds the same products in the same order."""
    import burn_dragon_amd as bda
    from burn_dragon_amd.kernel import relu_lowrank

    g = torch.Generator(device=DEV).manual_seed(d + N)
    x = torch.randn((B, h, T, d), device=DEV, generator=g)
    w = torch.randn((h, d, N), device=DEV, generator=g)
    bias = torch.randn((h, 1, N), device=DEV, generator=g)
    gate = torch.randn((B, h, T, N), device=DEV, generator=g)
    layout = bda.BlockPattern1d.from_blocks(16, list(range(0, (N + 15) // 16, 2)))
    ctx = bda.ffi.default_context(0)
    call = lambda: relu_lowrank.fused_forward(x, w, bias, 0.25, layout, gate=gate)
    try:
        ctx.set_option("relu_lowrank.row", 0)
        got = call()
        ctx.set_option("relu_lowrank.mfma_rows", 0)
        assert torch.equal(got, call())
    finally:
        ctx.set_option("relu_lowrank.mfma_rows", 2)
        ctx.set_option("relu_lowrank.row", 1)


@pytest.mark.parametrize("B,mult", [(17, 130), (33, 64), (16, 64)])
def test_encoder_of_a_batch_in_parts_of_several_k_blocks(B, mult):
    """The form with one chain per k-block of 1024, d = 512: 32 rows a tile with two k-blocks (the last part holding one) and
    with one k-block a workgroup, 16 rows a tile.  Against the VALU kernel: 2^-24 per step of a few dozen steps, 1e-5."""
    import burn_dragon_amd as bda

    d, V = 512, 64
    cfg = bda.BDHConfig(n_layer=1, n_embd=d, n_head=1, mlp_internal_dim_multiplier=mult, vocab_size=V)
    cfg.fused_kernels.set_rotary_embedding(bda.RotaryEmbedding.ALIBI)
    model = bda.BDH(cfg, DEV, seed=3)
    g = torch.Generator(device=DEV).manual_seed(B)
    tokens = torch.randint(0, V, (B, 1), device=DEV, generator=g)
    rho = torch.empty((1, B, 1, mult * d, d), device=DEV)
    rho.normal_(0.0, 0.1, generator=g)
    ctx = bda.ffi.default_context(0)
    logits = []
    try:
        for rows in (-16, 1 << 30):
            ctx.set_option("decoder.splitk_rows", rows)
            state = model.init_state()
            state.position, state.storage = 9, rho.clone()
            state.layers[0].rho = state.storage[0]
            logits.append(model.forward_with_state(tokens, state))
    finally:
        ctx.set_option("decoder.splitk_rows", 24)
    assert not torch.equal(logits[0], logits[1])
    assert rel_err(logits[0], logits[1]) < 1e-5


@pytest.mark.parametrize("B,d,h,mult", [(2, 128, 4, 4), (3, 256, 4, 8), (7, 68, 2, 3), (5, 512, 8, 8), (9, 256, 4, 72), (8, 192, 4, 65)])
def test_encoder_of_a_few_sequences_keeps_the_bits_of_the_valu_kernel(B, d, h, mult):
    """Two sequences and more of a small E, eight and more of a large one with d <= 256, on the f32 matrix cores."""
    import burn_dragon_amd as bda

    V = 64
    cfg = bda.BDHConfig(n_layer=1, n_embd=d, n_head=h, mlp_internal_dim_multiplier=mult, vocab_size=V)
    cfg.fused_kernels.set_rotary_embedding(bda.RotaryEmbedding.ALIBI)
    model = bda.BDH(cfg, DEV, seed=3)
    g = torch.Generator(device=DEV).manual_seed(B)
    tokens = torch.randint(0, V, (B, 1), device=DEV, generator=g)
    rho = 0.1 * torch.randn((1, B, h, mult * d // h, d), device=DEV, generator=g)
    ctx = bda.ffi.default_context(0)
    logits, names = [], []
    ctx.set_option("model.one_launch", 0)
    try:
        for rows in (24, 1 << 30):
            ctx.set_option("decoder.splitk_rows", rows)
            state = model.init_state()
            state.position, state.storage = 9, rho.clone()
            state.layers[0].rho = state.storage[0]
            with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
                logits.append(model.forward_with_state(tokens, state))
                torch.cuda.synchronize()
            names.append(" ".join(e.key for e in prof.key_averages()))
    finally:
        ctx.set_option("decoder.splitk_rows", 24)
        ctx.set_option("model.one_launch", 1)
    assert "k_decoder_rows" in names[0] and "k_decoder_rows" not in names[1]
    assert torch.equal(logits[0], logits[1])


@pytest.mark.parametrize("huge", ["embed", "decoder", "state"])
@pytest.mark.parametrize("d,h,N,V", [(128, 2, 64, 64), (260, 1, 64, 33)])
def test_two_launch_layer_norms_of_rows_whose_variance_is_no_float(huge, d, h, N, V):
    """A row whose variance is infinite is zero (c / inf), in the embedding, the encoder or the readout: the same values as
    kernel by kernel, and nothing that is no number."""
    import burn_dragon_amd as bda

    B = 3
    cfg = bda.BDHConfig(n_layer=2, n_embd=d, n_head=h, mlp_internal_dim_multiplier=1, vocab_size=V, dropout=0.0)
    cfg.latent_per_head = lambda: N
    cfg.fused_kernels.set_rotary_embedding(bda.RotaryEmbedding.ROPE)
    g = torch.Generator(device=DEV).manual_seed(d)
    w = {"embed": torch.randn((V, d), device=DEV, generator=g)}
    for name, shape in (("encoder", (h, d, N)), ("encoder_v", (h, d, N)), ("decoder", (h * N, d)), ("lm_head", (d, V))):
        w[name] = 0.05 * torch.randn(shape, device=DEV, generator=g)
    if huge == "embed":
        w["embed"][1] *= 1e20  # one sequence's row
    elif huge == "decoder":
        w["decoder"] *= 1e24
    model = bda.BDH(cfg, DEV, weights=w)
    start = torch.randn((2, B, h, N, d), device=DEV, generator=g) * (1e22 if huge == "state" else 0.1)
    tokens = torch.tensor([[0], [1], [2]], device=DEV)
    ctx = bda.ffi.default_context(0)
    logits, after = [], []
    try:
        for form in (1, 0):
            ctx.set_option("model.one_launch", form)
            state = model.init_state()
            state.position, state.storage = 5, start.clone()
            for i, layer in enumerate(state.layers):
                layer.rho = state.storage[i]
            logits.append(model.forward_with_state(tokens, state))
            after.append(state.storage)
    finally:
        ctx.set_option("model.one_launch", 1)
    torch.cuda.synchronize()
    assert torch.isfinite(logits[1]).all() and torch.isfinite(after[1]).all()
    assert rel_err(logits[0], logits[1]) < 1e-5
    assert rel_err(after[0], after[1]) < 1e-5


@pytest.mark.parametrize("form", ["model.one_launch", "model.fused_rows"])
@pytest.mark.parametrize("d,h,N", [(256, 4, 2048), (512, 4, 4096)])
def test_neurons_that_fire_in_one_form_of_a_decode_step_only_are_at_the_threshold(form, d, h, N):
    """The fused forms add D_x, and the sums behind its input row, in other orders than the kernels one by one.  Whether a neuron
    fires may differ only where its pre-activation p, here in float64, is within what rounding does to it: (d + 64) 2^-24
    sum |row w| for the chain of d terms and the LayerNorm of its row, and 1e-5 |row| |w|, by which the rows of two forms may
    differ, behind a layer.  Seen from the state: at position 0 a row of it that was zero is x v."""
    import burn_dragon_amd as bda

    N = 64 * 64 // h if form == "model.one_launch" else N  # ... which takes the two-launch layer up to 64 blocks of 64 neurons
    model = _model_of(d, h, N, layers=2)
    w = {k: t.double() for k, t in model.params.items()}
    g = torch.Generator(device=DEV).manual_seed(N)
    start = torch.zeros((2, 1, h, N, d), device=DEV)
    start[0, ..., : d // 2] = 0.1 * torch.randn((h, N, d // 2), device=DEV, generator=g)  # the other half shows what fired
    ctx, fired, ran = bda.ffi.default_context(0), [], []
    norm = lambda r: torch.nn.functional.layer_norm(r, (d,), eps=1e-5)
    for on in (1, 0):
        ctx.set_option(form, on)
        try:
            state = model.init_state()
            state.position, state.storage = 0, start.clone()
            for i, layer in enumerate(state.layers):
                layer.rho = state.storage[i]
            model.forward_with_state(torch.tensor([[5]], device=DEV), state)
            ran.append(_kernels_of_a_step(model, 1))
        finally:
            ctx.set_option(form, 1)
        fired.append((state.storage[:, 0, ..., d // 2:] != 0).any(-1))
    assert ran[0] != ran[1]
    row = norm(w["embed"][5])
    for l in range(2):
        p = torch.einsum("k,hkn->hn", row, w["encoder"])
        bound = (d + 64) * 2.0 ** -24 * torch.einsum("k,hkn->hn", row.abs(), w["encoder"].abs())
        if l:
            bound += 1e-5 * row.norm() * w["encoder"].norm(dim=1)
        for f in fired:
            assert bool(((f[l] == (p > 0)) | (p.abs() <= bound)).all()), l
        assert float((p.abs() <= bound).double().mean()) < 0.01 and 0.3 < float(fired[0][l].double().mean()) < 0.7
        x = p.clamp_min(0)
        attn = torch.einsum("hn,hnd->hd", x, start[l, 0].double())
        y = torch.einsum("hk,hkn->hn", norm(attn), w["encoder_v"]).clamp_min(0)
        row = norm(row + norm(torch.einsum("n,nd->d", (x * y).reshape(-1), w["decoder"])))


def _model_of(d, h, N, layers=1, rotary="rope", dtype="f32", lazy=False, vocab=64):
    import burn_dragon_amd as bda
    from burn_dragon_amd import ffi

    cfg = bda.BDHConfig(n_layer=layers, n_embd=d, n_head=h, mlp_internal_dim_multiplier=1, vocab_size=vocab, dropout=0.0)
    cfg.latent_per_head = lambda: N
    cfg.fused_kernels.set_rotary_embedding(bda.RotaryEmbedding.parse(rotary))
    g = torch.Generator(device=DEV).manual_seed(d + N)
    w = {"embed": torch.randn((vocab, d), device=DEV, generator=g)}
    for name, shape in (("encoder", (h, d, N)), ("encoder_v", (h, d, N)), ("decoder", (h * N, d)), ("lm_head", (d, vocab))):
        w[name] = 0.05 * torch.randn(shape, device=DEV, generator=g)
    return bda.BDH(cfg, DEV, weights=w, alibi_lazy=lazy, rho_dtype=ffi.BF16 if dtype == "bf16" else ffi.F32)


def _kernels_of_a_step(model, B):
    state = model.init_state()
    model._ensure_state(state, B)
    state.position = 3
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        model.forward_with_state(torch.zeros((B, 1), device=DEV, dtype=torch.int64), state)
        torch.cuda.synchronize()
    return " ".join(e.key for e in prof.key_averages())


@pytest.mark.parametrize("d,h,N,layers,kind,most,other", [
    (128, 4, 128, 4, ("rope", "f32", False), 128, "k_model_step"),     # 3 MiB of weights: a workgroup per sequence behind it
    (192, 4, 192, 4, ("rope", "f32", False), 81, "k_model_step"),      # 6.75 MiB
    (192, 4, 192, 4, ("pope", "f32", False), 121, "k_model_step"),     # every row visited whatever fires
    (256, 4, 256, 4, ("rope", "f32", False), 96, "k_decoder"),         # 3 MiB a layer
    (256, 4, 256, 4, ("alibi", "f32", False), 127, "k_model_step"),
    (256, 4, 256, 4, ("rope", "bf16", False), 64, "k_decoder"),
    (256, 4, 256, 4, ("alibi", "bf16", True), 126, "k_decoder"),
    (512, 8, 256, 2, ("rope", "bf16", False), 16, "k_decoder"),
    (384, 4, 384, 2, ("rope", "f32", False), 32, "k_decoder"),         # work for 512 columns
    (128, 4, 1024, 2, ("rope", "f32", False), 64, "k_decoder"),
    (192, 4, 96, 4, ("rope", "f32", False), 80, "k_model_step"),       # an odd number of blocks of 32
    (384, 4, 288, 2, ("rope", "f32", False), 28, "k_decoder"),
])
def test_where_the_two_launch_layer_ends(d, h, N, layers, kind, most, other):
    """The batch from which on another form is faster where few of the neurons fire."""
    rotary, dtype, lazy = kind
    model = _model_of(d, h, N, layers, rotary, dtype, lazy)
    inside, outside = _kernels_of_a_step(model, most), _kernels_of_a_step(model, most + 1)
    assert "k_layer_phase_a" in inside and "k_layer_phase_b" in inside
    assert "k_layer_phase" not in outside and other in outside


@pytest.mark.parametrize("d,h,N,first", [
    (512, 8, 512, 2),     # 8 MiB
    (512, 8, 576, 12),    # 9 MiB
    (512, 8, 1088, 24),   # 17 MiB
    (256, 4, 2052, 3),    # a little over 8 MiB
    (256, 4, 4096, 3),    # 16 MiB
    (256, 4, 4100, 8),
    (256, 4, 8192, 8),    # 32 MiB
    (256, 4, 8196, 24),
    (128, 4, 17000, 8),
])
def test_where_the_encoder_of_a_batch_takes_the_matrix_cores(d, h, N, first):
    """Below this batch the kernel that skips the rows of inactive neurons is the faster one where few of them fire."""
    import burn_dragon_amd as bda

    model = _model_of(d, h, N, rotary="alibi")
    ctx = bda.ffi.default_context(0)
    ctx.set_option("model.one_launch", 0)
    try:
        below, there = _kernels_of_a_step(model, first - 1), _kernels_of_a_step(model, first)
    finally:
        ctx.set_option("model.one_launch", 1)
    assert "k_decoder_partial" in below and "k_decoder_rows" not in below
    assert "k_decoder_rows" in there and "k_decoder_partial" not in there
