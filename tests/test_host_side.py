"""The library's host side on the CPU, over a stand-in for HIP's host calls (tests/hip_model.cpp): what
it queues where, and what it waits for."""

import pytest

import hip_model


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    return hip_model.build(tmp_path_factory.mktemp("hip_model"))


def test_memory_is_clear_before_anything_is_written_to_it(model):
    """hipMemset may return before its fill has run, and the context's stream does not wait for the null
    stream: a fill still on its way would take back what a write or a copy put there."""
    hip_model.run(model, """
        src, dst = rt.Memory(ctx, 4096), rt.Memory(ctx, 4096)
        data = np.arange(1024, dtype=np.uint32)
        src.write(data)
        rt.copy_regions(ctx, dst, src, [(0, 2048, 1024)])
        model.hip_model_settle()
        assert np.array_equal(src.read(np.uint32, 1024), data)
        want = np.zeros(1024, np.uint32)
        want[512:768] = data[:256]
        assert np.array_equal(dst.read(np.uint32, 1024), want)
        assert model.hip_model_violations() == 0
    """)


def test_a_prefills_tensors_are_clear_before_its_rows_are_copied_in(model):
    """The first prefill and each longer one allocate the tensors and clear them."""
    hip_model.run(model, """
        from tgx.synth import StackSpec
        spec = StackSpec(layers=1, dtype="bf16")
        shape = tgx.Shape(hidden=spec.hidden, inner=spec.inner, heads=spec.heads, kv_heads=spec.kv_heads,
                          head_dim=spec.head_dim, layers=1, capacity=640)
        dec = tgx.Decoder(ctx, shape, tgx.Batch(rows=1, slots=1))
        for n in (3, 300, 600):
            dec.prefill(0, np.ones((n, spec.hidden), np.float32))
        assert model.hip_model_violations() == 0
    """)


def test_a_models_tensors_are_clear_when_it_is_created(model):
    """No clear is left to run beside a new model's first copies and kernels."""
    hip_model.run(model, """
        from tgx.patch import Encoder, LmSide, PatchShape, Sampler
        shape, patch = tgx.Shape(layers=1, capacity=64), PatchShape(64, 4, 2, 1)
        kept = []  # destroying one waits for the device
        for create in (lambda: tgx.Decoder(ctx, shape, tgx.Batch(rows=1, slots=1)), lambda: Sampler(ctx, shape, patch),
                       lambda: Encoder(ctx, shape, patch), lambda: LmSide(ctx, shape, shape, tgx.Batch(rows=1, slots=1))):
            kept.append(create())
            assert model.hip_model_pending() == 0 and model.hip_model_violations() == 0, type(kept[-1])
    """)


@pytest.mark.parametrize("inner", [1024, 4096])
def test_a_gate_up_takes_the_grid_named_for_it_by_128s_of_tokens(model, inner):
    """A caller that names local_gate_up's grid as it was first cut (past 64 tokens a workgroup to 64
    columns and 128 tokens where the padded tokens come in 128s, else 64) is served whatever the kernel
    takes; another grid is refused."""
    hip_model.run(model, f"""
        inner = {inner}
        w = rt.Memory(ctx, 2 * inner * 1024 * 2)
        for tokens in (17, 64, 65, 128, 192, 256, 320, 345, 384, 700):
            pad = -(-tokens // 64) * 64 if tokens > 64 else -(-tokens // 16) * 16
            x, sq, mlp = rt.Memory(ctx, pad * 1024 * 2), rt.Memory(ctx, pad * 16 * 4), rt.Memory(ctx, pad * inner * 2)
            c = [tokens, 1, 1024, inner, 16, 2, rt.f32_bits(1e-5), 1]
            step = 128 if pad % 128 == 0 else 64
            first = (inner // 64, pad // step, 1) if tokens > 64 else (inner // 16, 1, 1)
            for groups in ((0, 0, 0), first):
                rt.dispatch(ctx, "local_gate_up", [x, w, sq, mlp], c, groups)
            try:
                rt.dispatch(ctx, "local_gate_up", [x, w, sq, mlp], c, (inner // 64, 40, 1))
            except tgx.TgxError as e:
                assert e.kind == "shape"
            else:
                assert False, tokens
    """)


@pytest.mark.parametrize("head_dim,capacity", [(64, 1152), (64, 2048), (128, 512), (128, 1024)])
def test_no_step_records_a_program(model, head_dim, capacity):
    """The programs of a decoder's rows are recorded when the rows are set, for steps with a row past
    decode_far positions and without: recording waits for everything queued on the context. A capacity
    that no such row fits has the one kind of program."""
    hip_model.run(model, f"""
        D, cap = {head_dim}, {capacity}
        line = 1152 if D == 64 else 512
        layers, h = 2, 1024 if D == 64 else 2048
        dec = tgx.Decoder(ctx, tgx.Shape(hidden=h, inner=4 * h if h == 1024 else 6144, head_dim=D, layers=layers, capacity=cap),
                          tgx.Batch(rows=2, slots=2))
        recorded = model.hip_model_graphs()
        assert recorded == (4 if cap > line else 2)
        x = np.zeros((2, h), np.float32)
        for position in [p for p in (0, line - 1, line, cap - 1, 0) if p < cap]:
            dec.step_rows([tgx.Row(position, 0), None], x)
            assert model.hip_model_last_nodes() == (6 if position >= line else 5) * layers + 1, position
        for at in [p for p in (0, line - 2, cap - 3, 0) if p + 2 < cap]:
            dec.set_rows([tgx.Row(at, 0), None], x)
            dec.launch(3, advance=True)
            dec.wait()
            assert model.hip_model_last_nodes() == (6 if at + 2 >= line else 5) * layers + 1, at
        assert model.hip_model_graphs() == recorded
    """)


@pytest.mark.parametrize("kv", [(2, 2), (2, 4)])
def test_no_step_of_the_lm_side_records_a_program(model, kv):
    """As above for both LMs at once, alone and in a patch step of fewer rows: at 20 rows an LM of 4 KV
    heads (80 groups) has its line at 4096 positions, one of 2 at 1152."""
    hip_model.run(model, f"""
        from tgx.patch import Encoder, LmSide, PatchShape, PatchStep, Sampler
        from tgx.synth import StackSpec, sampler_weights
        kv, rows, C, F = {kv}, 20, 64, 4
        lm = lambda kv: tgx.Shape(layers=1, kv_heads=kv, capacity=5000)
        side = LmSide(ctx, lm(kv[0]), lm(kv[1]), tgx.Batch(rows=rows, slots=rows))
        local, patch = tgx.Shape(layers=1, capacity=64), PatchShape(C, F, 2, rows)
        sampler, encoder = Sampler(ctx, local, patch), Encoder(ctx, local, patch)
        sampler.load_all(sampler_weights(StackSpec(layers=1, hidden=1024, inner=4096, dtype="bf16"), C))
        step = PatchStep(encoder, side, sampler)
        zeros = lambda *n: np.zeros(n, np.float32)
        at = lambda n, position: [tgx.Row(position if r == 0 else 3, r) for r in range(n)]
        for n in (rows, 3):
            step.run_rows(at(n, 0), zeros(n, C, F), zeros(n, C, F), zeros(n, 2))
            recorded = model.hip_model_graphs()
            for position in (1151, 1152, 4096, 0):
                step.run_rows(at(n, position), zeros(n, C, F), zeros(n, C, F), zeros(n, 2))
                assert model.hip_model_graphs() == recorded, (n, position)
        side.step_rows(at(rows, 0), zeros(rows, 1024))
        recorded = model.hip_model_graphs()
        for position in (1151, 1152, 4095, 4096, 0):
            side.step_rows(at(rows, position), zeros(rows, 1024))
            far = [position >= (4096 if rows * k > 64 else 1152) for k in kv]
            assert model.hip_model_last_nodes() == 8 + sum(7 if f else 6 for f in far), position
        for position in (1150, 4094):
            side.set_rows(at(rows, position), zeros(rows, 1024))
            side.launch(3, advance=True)
            side.wait()
            far = [position + 2 >= (4096 if rows * k > 64 else 1152) for k in kv]
            assert model.hip_model_last_nodes() == 8 + sum(7 if f else 6 for f in far), position
        assert model.hip_model_graphs() == recorded
    """)


@pytest.mark.parametrize("N", [16, 48, 1008, 1024, 1040])
@pytest.mark.parametrize("rows", [1, 2, 17])
def test_a_residuals_next_input_holds_its_last_half_block(model, N, rows):
    """gemv_residual writes out_n in blocks of 32 columns, a row's 32 after another row's: where N ends
    in half a block, the last row's half lies past rows x N. The bytes written up to it are what the
    binding must hold, and no more."""
    hip_model.run(model, f"""
        N, rows, K = {N}, {rows}, 1024
        last = max((n // 32 * rows + b) * 32 + n % 32 for n in range(N) for b in range(rows))
        full = rt.Memory(ctx, 1 << 22)
        c = [1024, 4096, 16, 2, rows, 64, rows, 1, rows, rt.f32_bits(1e-5), 1, 64, K, N, 4]
        for short in (0, 2):
            out_n = rt.Memory(ctx, 2 * (last + 1) - short)
            try:
                rt.dispatch(ctx, "gemv_residual", [full, full, full, full, full, out_n, full], c)
            except tgx.TgxError as e:
                assert short and e.kind == "shape" and "out_n" in str(e), str(e)
            else:
                assert not short
    """)
