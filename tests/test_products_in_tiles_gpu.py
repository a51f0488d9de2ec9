"""Products in tiles (csrc/hip/gemm_tiles.hip): every tile at the sizes where its edges, its ring of stages and its slices of K
can go wrong, against products in 64 bits, and the rule that hands products of many rows to it."""
import ctypes as C
import functools

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from kvcm_amd import ops as _ops
    _ops.lib()
    return _ops


def _tiles(ops):
    out = []
    for t in range(ops.lib().kvcm_gemm_tiles_count()):
        bm, bn = C.c_int(), C.c_int()
        assert ops.lib().kvcm_gemm_tiles_size(t, C.byref(bm), C.byref(bn)) == 0
        out.append((bm.value, bn.value))
    return out


def _operands(seed, M, N, K, pad_x=0, pad_w=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(M, K + pad_x, generator=g, device=DEV).to(torch.bfloat16)[:, :K]
    w = (torch.randn(N, K + pad_w, generator=g, device=DEV) * 0.1).to(torch.bfloat16)[:, :K]
    return x, w


def _close(got, x, w, bf16, ref=None):
    """32-bit sums in any order are off by at most K 2^-24 of the sum of the terms' sizes each (two operations a term counted);
    a bfloat16 result by half a unit of its own last place beside that."""
    xd, wd = x.double(), w.double()
    ref = xd @ wd.t() if ref is None else ref
    bound = 2 * x.shape[1] * 2.0 ** -24 * (xd.abs() @ wd.abs().t())
    if bf16:
        bound = bound + ref.abs() * 2.0 ** -8
    err = (got.double() - ref).abs()
    assert bool((err <= bound).all()), float((err - bound).max())


def _run(ops, x, w, partials, out, S=1, gated=0, act=0, limit=0.0, tile=-1, N=None):
    M, K = x.shape
    N = N or w.shape[0]
    rc = ops.lib().kvcm_gemm_tiles(x.data_ptr(), w.data_ptr(), partials.data_ptr() if partials is not None else 0, out.data_ptr(),
                                   ops._DT[out.dtype], M, N, K, x.stride(0), w.stride(0), out.stride(0), S, gated, act, limit,
                                   tile, ops._stream())
    assert rc == 0, ops.lib().kvcm_hip_last_error().decode()


@pytest.mark.parametrize("tile", range(17))
def test_every_tile_at_its_edges(ops, tile):
    sizes = _tiles(ops)
    assert len(sizes) == 17
    bm, bn = sizes[tile]
    seed = 0
    # rows and columns around one tile and around several; k of one step (shorter than any ring), of few, of more than a ring
    for M, N, K, S in [(1, 64, 64, 1), (bm - 1, bn, 448, 1), (bm + 1, bn + 12, 640, 2), (2 * bm + 3, 2 * bn - 4, 192, 3),
                       (5, 4 * bn + 64, 1152, 4), (bm, 8, 576, 8), (3 * bm, 3 * bn, 128, 1)]:
        seed += 1
        x, w = _operands(seed, M, N, K, pad_x=8 * (seed % 3), pad_w=8 * (seed % 2))
        if S > 1:
            parts = torch.full((S * M * N + 4,), float("nan"), device=DEV)
            _run(ops, x, w, parts, torch.empty(M, N, device=DEV), S=S, tile=tile)
            assert torch.isnan(parts[S * M * N:]).all()
            _close(parts[:S * M * N].view(S, M, N).double().sum(0), x, w, False)
            continue
        for dtype, pad in ((torch.float32, 0), (torch.float32, 3), (torch.bfloat16, 0), (torch.bfloat16, 5)):
            room = torch.full((M * (N + pad) + 9,), float("nan"), dtype=dtype, device=DEV)
            out = room[1:1 + M * (N + pad)].view(M, N + pad)[:, :N]      # begins at any element
            _run(ops, x, w, None, out, tile=tile)
            _close(out, x, w, dtype == torch.bfloat16)
            left = room.clone()
            left[1:1 + M * (N + pad)].view(M, N + pad)[:, :N] = float("nan")
            assert torch.isnan(left).all(), "written beside the result"


@pytest.mark.parametrize("tile", range(17))
def test_every_tile_gated(ops, tile):
    bm, bn = _tiles(ops)[tile]
    for seed, (M, I, K) in enumerate([(1, 8, 64), (bm + 1, bn // 2, 448), (bm - 1, bn + 8, 640), (2 * bm + 3, 2 * bn + 40, 192)]):
        x, w = _operands(50 + seed, M, 2 * I, K)
        g, u = (x.double() @ w.double().t()).split(I, 1)
        size = 2 * K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
        eg, eu = size.split(I, 1)
        exact = g * torch.sigmoid(g) * u
        # d silu <= 1.1 d gate; silu by the hardware's exp2 and reciprocal: 2^-21 of itself
        bound = 1.1 * eg * u.abs() + g.abs() * eu + 1.1 * eg * eu + exact.abs() * 2.0 ** -21
        for dtype in (torch.float32, torch.bfloat16):
            out = torch.full((M, I), float("nan"), dtype=dtype, device=DEV)
            _run(ops, x, w, None, out, gated=1, act=1, tile=tile, N=I)
            last = exact.abs() * 2.0 ** -8 if dtype == torch.bfloat16 else 0
            assert bool(((out.double() - exact).abs() <= bound + last).all())
        _run(ops, x, w, None, out, gated=1, act=2, tile=tile, N=I)
        relu = g.clamp(min=0) * u
        assert bool(((out.double() - relu).abs() <= eg * u.abs() + g.abs() * eu + eg * eu + relu.abs() * 2.0 ** -8).all())
        # with a stored product's roundings: what the product stored in bfloat16 gives through the SwiGLU launch, but for sums that round to the other side
        out = torch.full((M, I), float("nan"), dtype=torch.bfloat16, device=DEV)
        _run(ops, x, w, None, out, gated=1, act=0, tile=tile, N=I)
        gu, want = torch.empty(M, 2 * I, dtype=torch.bfloat16, device=DEV), torch.empty_like(out)
        _run(ops, x, w, None, gu, tile=tile)
        ops.swiglu(gu, want)
        assert (out == want).float().mean() > 0.98
        # gate (d silu <= 1.1 d gate), silu(gate), up and the result are rounded to bfloat16, by at most 2^-8 of themselves each
        assert bool(((out.double() - exact).abs() <= 1.1 * bound + 4.2 * 2.0 ** -8 * g.abs() * u.abs()).all())
        _run(ops, x, w, None, out, gated=1, limit=0.5, tile=tile, N=I)
        gc, uc = g.clamp(max=0.5), u.clamp(-0.5, 0.5)
        clamped = gc * torch.sigmoid(1.702 * gc) * (uc + 1)
        assert bool(((out.double() - clamped).abs() <= 2.5 * (eg + eu) + clamped.abs() * 2.0 ** -8 + 1e-6).all())


def test_products_with_a_folded_norm_in_tiles(ops):
    """rows whose norm's scale is applied to the sums: rsqrt(mean x^2 + eps) from sums of squares of 8 columns each"""
    M, I, K = 8, 8192 + 64, 320
    x, w = _operands(90, M, 2 * I, K)
    ss = torch.rand(M, K // 8, device=DEV) * 8
    rstd = 1.0 / torch.sqrt(ss.double().sum(1, keepdim=True) / K + 1e-5)
    out = torch.empty(M, I, dtype=torch.bfloat16, device=DEV)
    assert ops.lib().kvcm_gemm_skinny_swiglu_normed(x.data_ptr(), w.data_ptr(), ss.data_ptr(), K // 8, 1e-5, out.data_ptr(), M, I, K,
                                                    x.stride(0), w.stride(0), out.stride(0), ops._stream()) == 0
    g, u = (x.double() @ w.double().t() * rstd).split(I, 1)
    want = g * torch.sigmoid(g) * u
    # gate (d silu <= 1.1 d gate), silu(gate), up and the result are rounded to bfloat16, by at most 2^-8 of themselves each
    assert bool(((out.double() - want).abs() <= 4.2 * 2.0 ** -8 * (g.abs() * u.abs()) + 1e-5).all())


def _apart(t, ld):
    """the same rows, ld elements apart"""
    room = torch.empty((t.shape[0] - 1) * ld + t.shape[1], dtype=t.dtype, device=t.device)
    out = room.as_strided(t.shape, (ld, 1))
    out.copy_(t)
    return out


# ld: the first that a tile's 32-bit offsets are not meant for; rows so far apart that offsets inside a tile pass 32 bits
@pytest.mark.parametrize("M,N,K,ld", [(5, 64, 128, 1 << 22), (40, 128, 256, 1 << 22), (40, 64, 640, 1 << 26), (200, 64, 128, 1 << 22)])
def test_rows_far_apart(ops, M, N, K, ld):
    lib, x, w = ops.lib(), *_operands(M + N, M, N, K)
    for far_x, far_w in ((_apart(x, ld), w), (x, _apart(w, ld)), (_apart(x, ld), _apart(w, ld))):
        ends = (far_x.data_ptr(), far_w.data_ptr()), (M, N, K, far_x.stride(0), far_w.stride(0), N)
        S = min(2, K // 64)
        parts, out = torch.empty(S, M, N, device=DEV), torch.full((M, N), float("nan"), device=DEV)
        assert lib.kvcm_gemm_skinny(*ends[0], parts.data_ptr(), 0, ops._DT[torch.float32], *ends[1], S, ops._stream()) == 0, lib.kvcm_hip_last_error()
        _close(parts.double().sum(0), x, w, False)
        assert lib.kvcm_gemm_skinny(*ends[0], 0, out.data_ptr(), ops._DT[torch.float32], *ends[1], 1, ops._stream()) == 0, lib.kvcm_hip_last_error()
        _close(out, x, w, False)
        if M < ops.LIBRARY_GEMM_MIN_ROWS:
            _close(ops.gemm(far_x, far_w, out.fill_(float("nan"))), x, w, False)


@pytest.mark.parametrize("M,I,K", [(40, 5120, 64), (3, 8192, 128)])
def test_gated_products_of_rows_far_apart(ops, M, I, K):
    x, w = _operands(M + I, M, 2 * I, K)
    far, out = _apart(x, 1 << 22), torch.empty(M, I, dtype=torch.bfloat16, device=DEV)
    ss = torch.rand(M, K // 8, device=DEV) * 8
    g, u = (x.double() @ w.double().t()).split(I, 1)
    rstd = 1.0 / torch.sqrt(ss.double().sum(1, keepdim=True) / K + 1e-5)
    at, to = (far.data_ptr(), w.data_ptr()), (M, I, K, far.stride(0), K, I)
    for scale in (1.0, rstd):
        out.fill_(float("nan"))
        if scale is rstd:
            rc = ops.lib().kvcm_gemm_skinny_swiglu_normed(*at, ss.data_ptr(), K // 8, 1e-5, out.data_ptr(), *to, ops._stream())
        else:
            rc = ops.lib().kvcm_gemm_skinny_swiglu(*at, out.data_ptr(), ops._DT[torch.bfloat16], *to, 0.0, ops._stream())
        assert rc == 0, ops.lib().kvcm_hip_last_error()
        want = g * scale * torch.sigmoid(g * scale) * u * scale
        # gate (d silu <= 1.1 d gate), silu(gate), up and the result are rounded to bfloat16, by at most 2^-8 of themselves each
        assert bool(((out.double() - want).abs() <= 4.2 * 2.0 ** -8 * (g * scale).abs() * (u * scale).abs() + 1e-5).all())


@pytest.mark.parametrize("M,N,K,mine", [(96, 2048, 2048, True), (200, 2560, 2048, True), (333, 2048, 5632, True), (700, 2048, 2048, False),
                                        (700, 512, 1024, True), (1024, 1536, 512, True), (640, 64, 14336, False), (2000, 256, 5632, False), (1536, 8192, 2048, False), (2000, 192, 128, None), (768, 2048, 5632, None), (1000, 192, 8192, None)])
def test_many_rows_go_to_the_tiles_where_the_rule_says_so(ops, M, N, K, mine):
    x, w = _operands(M, M, N, K)
    for dtype in (torch.bfloat16, torch.float32):
        out = torch.full((M, N), float("nan"), dtype=dtype, device=DEV)
        scratch = torch.empty(8 * 512 * N, device=DEV)
        S = ops.skinny_splits(M, N, K) if M <= 512 else 1
        if mine is not None:
            assert ops._tiles_take(M, N, K, S) == mine
        got = ops.gemm(x, w, out, scratch=scratch, keep_partial=True)
        _close(got.materialize() if isinstance(got, ops.PartialSums) else got, x, w, dtype == torch.bfloat16)
        _close(ops.gemm(x, w, out, scratch=scratch), x, w, dtype == torch.bfloat16)
    act, plain = torch.empty(M, N // 2, dtype=torch.bfloat16, device=DEV), torch.empty(M, N // 2, dtype=torch.bfloat16, device=DEV)
    assert ops.gemm_swiglu(x, w, act) == ops._tiles_take(M, N // 2, K, 1, gated=True)
    if ops._tiles_take(M, N // 2, K, 1, gated=True):
        ops.swiglu(ops.gemm(x, w, torch.empty(M, N, dtype=torch.bfloat16, device=DEV)), plain)
        assert (act == plain).float().mean() > 0.98
        # gate (d silu <= 1.1 d gate), silu(gate), up and the result are rounded to bfloat16, by at most 2^-8 of themselves each
        g, u = (x.double() @ w.double().t()).split(N // 2, 1)
        assert bool(((act.double() - g * torch.sigmoid(g) * u).abs() <= 4.2 * 2.0 ** -8 * g.abs() * u.abs() + 1e-4).all())


@pytest.mark.parametrize("tile", range(7))
def test_routed_experts_in_every_tile(ops, tile, monkeypatch):
    """groups that end inside a tile, in several tiles of an expert, K that ends inside a step, columns that end inside a tile"""
    import test_routed_forms_gpu as forms
    assert ops.lib().kvcm_moe_grouped_tile_count() == 7
    monkeypatch.setattr(ops, "moe_grouped", functools.partial(ops.moe_grouped, tile_up=tile, tile_down=(tile + 3) % 7))
    for T, E, top, K, F, H, kind, one in forms.GROUPED + [(700, 3, 2, 320, 208, 516, "silu", False)]:
        chosen = torch.zeros(T, top, dtype=torch.long) if one else None
        forms._check("grouped", forms._case(T, E, top, K, F, H, kind, T + K, chosen), kind, tile % 2 == 0, tile % 2 == 1)


@pytest.mark.parametrize("M,I,K,one", [(1, 2816, 2048, False), (2, 2560, 2048, True), (8, 2048, 2048, False), (9, 512, 2048, True), (95, 512, 2112, False),
                                       (300, 1408, 2048, True), (1, 5120, 64, True), (40, 2816, 8, False)])
def test_gated_products_without_roundings_before_the_end(ops, M, I, K, one):
    """the rule, and each activation as ``gated_act`` of the product's 32-bit result gives it"""
    x, w = _operands(M + I, M, 2 * I, K)
    gu = (x.double() @ w.double().t()).float()
    for activation, limit in (("relu", 0.0), ("silu", 0.0), ("clamped", 1.5)):
        got = torch.full((M, I), float("nan"), dtype=torch.bfloat16, device=DEV)
        assert ops.gemm_gated(x, w, got, activation, limit) == one
        if one:
            want = torch.empty_like(got)
            ops.gated_act(gu, want, activation, limit=limit)
            # both round once; 32-bit sums of K terms may fall on the other side of a tie
            scale = gu[:, :I].abs() * gu[:, I:].abs() + gu.abs().amax() * 2.0 ** -8
            assert (got == want).float().mean() > 0.98
            assert bool(((got.float() - want.float()).abs() <= 2.0 ** -7 * (scale + want.float().abs())).all())
    assert ops.gemm_gated(x, w, got, "gelu") is False and ops.gemm_gated(x.float(), w.float(), got.float(), "relu") is False


@pytest.mark.parametrize("M", [64, 200])
@pytest.mark.parametrize("activation,limit", [("silu", 0.0), ("clamped", 7.0), ("relu", 0.0)])
def test_gated_products_apply_the_exact_functions(ops, M, activation, limit):
    """sums of one term each are exact, so the product gives what ``gated_act`` gives for them, bit for bit: the hardware's exp2 and
    reciprocal, 2^-24 of the gate's size off, would fall on the other side of a tie here and there"""
    I, K = 1024, 64
    x, w = torch.zeros(M, K, device=DEV), torch.zeros(2 * I, K, device=DEV)
    x[:, 0], x[:, 1] = torch.linspace(-60.0, 8.0, M, device=DEV), 1.0
    w[:I, 0], w[I:, 1] = torch.linspace(0.25, 1.0, I, device=DEV), torch.linspace(-3.0, 5.0, I, device=DEV)
    x, w = x.to(torch.bfloat16), w.to(torch.bfloat16)
    got, want = (torch.full((M, I), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(2))
    assert ops.gemm_gated(x, w, got, activation, limit)
    ops.gated_act((x.double() @ w.double().t()).float(), want, activation, limit=limit)
    assert torch.equal(got, want), int((got != want).sum())


def test_a_gate_with_limits_needs_a_limit(ops):
    x, w = _operands(7, 200, 1024, 64)
    got = torch.empty(200, 512, dtype=torch.bfloat16, device=DEV)
    assert ops.gemm_gated(x, w, got, "clamped", 1.0) and not ops.gemm_gated(x, w, got, "clamped", 0.0) and not ops.gemm_gated(x, w, got, "clamped")
    with pytest.raises(ops.KernelError, match="positive limit"):
        ops.gated_act(torch.zeros(200, 1024, device=DEV), got, "clamped")


def test_tuned_library_products_take_gate_and_up_too(ops, tmp_path, monkeypatch):
    """who asks for the library's tuned algorithms gets them for the largest product of a layer as for the others"""
    x, w = _operands(8, 128, 1024, 64)
    act = torch.empty(128, 512, dtype=torch.bfloat16, device=DEV)
    for mode in ("heuristic", "all"):
        assert not ops.gemm_swiglu(x, w, act, tuning=mode) and not ops.gemm_gated(x, w, act, tuning=mode)
        with monkeypatch.context() as m:
            m.setattr(ops, "LIBRARY_TUNING", mode)
            assert not ops.gemm_swiglu(x, w, act) and not ops.gemm_gated(x, w, act)
            assert ops.gemm_swiglu(x, w, act, tuning="off") and ops.gemm_gated(x, w, act, tuning="off")
        assert ops.gemm_gated(x[:64], w, act[:64], tuning=mode)      # (few rows are never the library's)
    assert ops.gemm_swiglu(x, w, act) and ops.gemm_gated(x, w, act)

    from kvcm_amd.config.engine_config import EngineConfig
    from kvcm_amd.config.model_config import LlamaConfig
    from kvcm_amd.engine.engine import Engine
    from kvcm_amd.weights.random_init import write_model_dir
    raw = dict(vocab_size=256, hidden_size=64, intermediate_size=320, num_hidden_layers=1, num_attention_heads=4, num_key_value_heads=2, head_dim=16,
               max_position_embeddings=256, rope_theta=10000.0, rms_norm_eps=1e-5, tie_word_embeddings=False)
    write_model_dir(str(tmp_path), "LlamaForCausalLM", LlamaConfig.from_dict(raw), seed=0, dtype=torch.float32)
    eng = Engine(str(tmp_path), EngineConfig(block_size=16, num_blocks=64, max_seq_len=256, max_num_seqs=2, max_batched_tokens=160, dtype="bfloat16",
                                             tune_products="heuristic"))
    before = len(ops.library_tuning_log)
    eng.generate([list(range(130))], max_new_tokens=1)
    assert (640, 64) in [entry[1:3] for entry in ops.library_tuning_log[before:]], ops.library_tuning_log[before:]
