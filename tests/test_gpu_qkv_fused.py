"""GPU: the QKV projection with its q/k RMSNorm, RoPE and KV-ring write in one op
(fp8_qkv_norm_rope_cache) equals the two-op sequence it replaces -- fp8_scaled_mm into a bf16
[M, 3*H*D] buffer, then fused_qkv_norm_rope_cache on that buffer (dit.py:409-451) -- bit for bit,
on every output: rotated Q and K, the ring slot's K (normalised or rotated) and V, the second V
destination, and the ring rows and slots it must not touch.

Cases cover the ways a row reaches the outputs: the persistent kernel's fused epilogue (from 7/8 of a
round of 256x256 tiles on), the sub-tiles of a last partial round (stored plainly, then the tail
kernel), the rows below whole rounds (a small GEMM, then the standalone kernel), and the two-op
sequence itself with fewer tiles and for shapes the epilogue does not take (odd head counts, head_dim
64, K % 256 != 0). Most operands are exact small integers with power-of-two scales, so every GEMM
output is exact whatever the summation order and the comparison isolates the norm/RoPE/ring work;
test_same_gemm_kernels_as_the_two_ops takes operands whose sums show the order.
"""
import numpy as np
import pytest
import torch

from gpu_util import DEV, announce, gen, kernels_of, u16
from oracle import rope as orope
from oracle.fp8 import f32_to_bf16, f32_to_e4m3fn

pytestmark = pytest.mark.gpu


def _fp8(a_f32: np.ndarray) -> torch.Tensor:
    return torch.from_numpy(f32_to_e4m3fn(a_f32)).view(torch.float8_e4m3fn).to(DEV)


def _bf16(a_f32: np.ndarray) -> torch.Tensor:
    return torch.from_numpy(f32_to_bf16(a_f32).view(np.int16)).view(torch.bfloat16).to(DEV)


def _problem(M, K, H, D, seed, exact):
    """Quantised activations [M, K], weight (K, N) column-major, scales, bias, norm weights and RoPE
    tables [M, D/2]."""
    rng = np.random.default_rng(seed)
    N = 3 * H * D
    if exact == "order":
        # positive products over 30 binary places in the first half of K, taken back but for a few per cent of them
        # in the second: the sums pass through 100 times their result, whose bf16 bits then show the order of adding
        x, y = (np.exp(1.5 * rng.standard_normal((r, K // 2))).clip(2.0 ** -8, 400).astype(np.float32) for r in (M, N))
        z = np.where(rng.random(y.shape) < 0.05, np.roll(y, 1, axis=1), y)
        a, w = _fp8(np.concatenate([x, -x], axis=1)), _fp8(np.concatenate([y, z], axis=1))
        sa = torch.from_numpy((2.0 ** rng.integers(-10, -5, M)).astype(np.float32)).to(DEV)
        sw = torch.from_numpy((2.0 ** rng.integers(-8, -4, N)).astype(np.float32)).to(DEV)
    elif exact:
        a = _fp8(rng.integers(-8, 9, (M, K)).astype(np.float32))
        w = _fp8(rng.integers(-8, 9, (N, K)).astype(np.float32))
        sa = torch.from_numpy((2.0 ** rng.integers(-10, -5, M)).astype(np.float32)).to(DEV)
        sw = torch.from_numpy((2.0 ** rng.integers(-8, -4, N)).astype(np.float32)).to(DEV)
    else:
        import joyomni_ops as jo
        g = gen(seed)
        x = torch.randn(M, K, generator=g).to(torch.bfloat16).to(DEV)
        wf = (0.05 * torch.randn(N, K, generator=g)).to(torch.bfloat16).to(DEV)
        a = torch.empty(M, K, dtype=torch.float8_e4m3fn, device=DEV)
        w = torch.empty(N, K, dtype=torch.float8_e4m3fn, device=DEV)
        sa = torch.empty(M, 1, device=DEV)
        sw = torch.empty(N, 1, device=DEV)
        jo.per_token_quant_fp8(x, a, sa, True)
        jo.per_token_quant_fp8(wf, w, sw, True)
        sa, sw = sa.reshape(M), sw.reshape(N)
    bias = _bf16((rng.integers(-32, 32, N) / 16).astype(np.float32))
    qw = _bf16((1 + 0.1 * rng.standard_normal(D)).astype(np.float32))
    kw = _bf16((1 + 0.1 * rng.standard_normal(D)).astype(np.float32))
    # 3-D RoPE tables of a frames x 16 x ww grid (at least M tokens), first M rows
    frames = max(1, M // 400)
    ww = (M + frames * 16 - 1) // (frames * 16)
    dims = (44, 42, 42) if D == 128 else (24, 20, 20)
    _, _, cb, sb = orope.rope_half_tables(list(range(frames)), 16, ww, dims, 10000.0)
    cos = torch.from_numpy(np.ascontiguousarray(cb[:M]).view(np.int16)).view(torch.bfloat16).to(DEV)
    sin = torch.from_numpy(np.ascontiguousarray(sb[:M]).view(np.int16)).view(torch.bfloat16).to(DEV)
    return a, w.t(), sa, sw, bias, qw, kw, cos, sin


def _outputs(M, H, D, slots, cap, seed):
    g = gen(seed)
    q = torch.randn(M, H, D, generator=g).to(torch.bfloat16).to(DEV)  # garbage: every row is written
    k = torch.randn(M, H, D, generator=g).to(torch.bfloat16).to(DEV)
    v = torch.randn(M, H, D, generator=g).to(torch.bfloat16).to(DEV)
    ck = torch.randn(slots, cap, H, D, generator=g).to(torch.bfloat16).to(DEV)  # other rows must keep these
    cv = torch.randn(slots, cap, H, D, generator=g).to(torch.bfloat16).to(DEV)
    return q, k, v, ck, cv


def _shift_table(t, elems):
    """The same table in a buffer whose first row starts `elems` elements past an aligned address."""
    buf = torch.empty(t.numel() + elems, dtype=t.dtype, device=t.device)
    view = buf[elems:].view(t.shape)
    view.copy_(t)
    return view


def _run_both(M, K, H, D, seed, exact, cache_tokens=-1, pre_rope=True, with_q=True, with_k=True, with_v=True,
              slot=1, offset=3, table_shift=0):
    import joyomni_ops as jo
    a, b, sa, sw, bias, qw, kw, cos, sin = _problem(M, K, H, D, seed, exact)
    if table_shift:
        cos, sin = _shift_table(cos, table_shift), _shift_table(sin, table_shift)
    n = M if cache_tokens < 0 else cache_tokens
    slots, cap = 3, offset + M + 5
    ref = _outputs(M, H, D, slots, cap, seed + 1)
    got = tuple(t.clone() for t in ref)
    y = jo.fp8_scaled_mm(a, b, sa, sw, torch.bfloat16, bias)
    jo.fused_qkv_norm_rope_cache(y, H, 1e-6, qw, kw, cos, sin, ref[0] if with_q else None, ref[1] if with_k else None,
                                 ref[3], ref[4], slot, offset, v_out=ref[2] if with_v else None, cache_tokens=n,
                                 cache_pre_rope=pre_rope)
    jo.fp8_qkv_norm_rope_cache(a, b, sa, sw, bias, H, 1e-6, qw, kw, cos, sin, got[0] if with_q else None,
                               got[1] if with_k else None, got[3], got[4], slot, offset,
                               v_out=got[2] if with_v else None, cache_tokens=n, cache_pre_rope=pre_rope)
    torch.cuda.synchronize()
    for name, r, o in zip(("q_out", "k_out", "v_out", "ring K", "ring V"), ref, got):
        assert torch.equal(u16_t(r), u16_t(o)), f"{name} differs ({M}x{K}, H {H}, D {D})"


def u16_t(t):
    return t.contiguous().view(torch.int16)


@pytest.mark.parametrize("M,K,H,D", [
    (4352, 1024, 32, 128),  # whole rounds through the fused epilogue + q, k and v tiles as quarter sub-tiles
    (2048, 1024, 8, 128),   # 96 tiles, less than 7/8 of a round: the two ops themselves
    (1000, 2048, 16, 128),  # the same, ragged M
    (777, 512, 5, 128),     # odd head count: the two ops
    (300, 1024, 6, 64),     # head_dim 64: the two ops
    (640, 640, 4, 128),     # K % 256 != 0: the two ops
    (1002, 1024, 8, 128),   # less than 7/8 of a round, M % 4 != 0
])
def test_exact_equals_gemm_then_norm_rope(M, K, H, D):
    announce("fp8 qkv norm rope exact", M, K, H, D)
    _run_both(M, K, H, D, M + K + H, exact=True)


@pytest.mark.parametrize("pre_rope", [True, False])
def test_partial_cache_and_post_rope_ring(pre_rope):
    """kv_cache_write_seq_len: only the first rows reach the ring (at an offset, in slot 1); the ring K
    before or after RoPE."""
    announce("fp8 qkv norm rope partial cache", pre_rope)
    _run_both(4352, 1024, 32, 128, 11, exact=True, cache_tokens=4000, pre_rope=pre_rope)


def test_cache_only_forward():
    """kv_cache_write_only: no Q / K / V outputs, only the ring."""
    announce("fp8 qkv norm rope cache only")
    _run_both(4352, 1024, 32, 128, 12, exact=True, with_q=False, with_k=False, with_v=False)


def test_block_shape_random_operands():
    """The block's video stream at the benchmark's size (10800 tokens, 40 x 128 heads, K 5120) on
    random quantised operands: the fused op and the two-op sequence give every row the same GEMM kernel,
    so every output is bit-identical (the whole rounds through the fused epilogue, the last round's
    V tiles as quarter sub-tiles)."""
    announce("fp8 qkv norm rope block shape", 10800, 5120, 40, 128)
    _run_both(10800, 5120, 40, 128, 13, exact=False)


@pytest.mark.parametrize("M", [4352, 4096])  # a partial last round; whole rounds (no scratch otherwise)
def test_tables_not_16_byte_aligned(M):
    """cos / sin rows that start 8 bytes past a 16-byte boundary: the torch op reads an aligned copy
    (fused epilogue), the same bits as the two-op sequence."""
    announce("fp8 qkv norm rope unaligned tables", M)
    _run_both(M, 1024, 32, 128, 14, exact=True, table_shift=4)


def test_capi_unaligned_tables_need_the_full_scratch():
    """Through the C ABI, misaligned tables send the call to the unfused path, which needs the whole
    [M, 3E] bf16 scratch even where the size query says 0 (4096 rows: whole rounds of tiles): with
    no scratch the call fails before any launch and leaves the outputs alone; with M x 3E x 2 bytes
    it gives the two-op sequence's bits."""
    import joyomni_ops as jo
    from joyomni_ops import _lib
    announce("fp8 qkv norm rope C ABI unaligned tables")
    M, K, H, D = 4096, 1024, 32, 128
    N = 3 * H * D
    a, b, sa, sw, bias, qw, kw, cos, sin = _problem(M, K, H, D, 16, exact=True)
    cos, sin = _shift_table(cos, 4), _shift_table(sin, 4)
    assert jo._LIB.joy_fp8_qkv_norm_rope_cache_scratch_size(M, K, H, D) == 0
    slots, cap = 2, M
    ref = _outputs(M, H, D, slots, cap, 17)
    got = tuple(t.clone() for t in ref)
    y = jo.fp8_scaled_mm(a, b, sa, sw, torch.bfloat16, bias)
    jo.fused_qkv_norm_rope_cache(y, H, 1e-6, qw, kw, cos, sin, ref[0], ref[1], ref[3], ref[4], 1, 0, v_out=ref[2])
    before = tuple(t.clone() for t in got)
    st = torch.cuda.current_stream().cuda_stream

    def call(scratch, nbytes):
        return jo._LIB.joy_fp8_qkv_norm_rope_cache(
            a.data_ptr(), b.data_ptr(), sa.data_ptr(), sw.data_ptr(), bias.data_ptr(), M, K, H, D, 1e-6,
            qw.data_ptr(), kw.data_ptr(), cos.data_ptr(), sin.data_ptr(), got[0].data_ptr(), H * D,
            got[1].data_ptr(), H * D, got[2].data_ptr(), H * D, got[3].data_ptr(), got[4].data_ptr(), slots, cap, 1,
            0, M, 0, scratch, nbytes, st)

    rc = call(None, 0)
    assert rc == 1, rc  # JOY_ERR_INVALID_ARGUMENT
    assert b"scratch needed for this call" in jo._LIB.joy_last_error()
    torch.cuda.synchronize()
    for r, o in zip(before, got):
        assert torch.equal(u16_t(r), u16_t(o)), "outputs written by a refused call"
    scratch = torch.empty(M * N * 2, dtype=torch.uint8, device=DEV)
    _lib.check(jo._LIB, call(scratch.data_ptr(), scratch.numel()))
    torch.cuda.synchronize()
    for name, r, o in zip(("q_out", "k_out", "v_out", "ring K", "ring V"), ref, got):
        assert torch.equal(u16_t(r), u16_t(o)), f"{name} differs"


def test_no_ring_rows_written():
    """cache_tokens = 0: the ring keeps every row; Q / K / V are still written."""
    announce("fp8 qkv norm rope no ring rows")
    _run_both(4352, 1024, 32, 128, 15, exact=True, cache_tokens=0)


@pytest.mark.parametrize("M", [515, 4353, 4354])  # a partial last tile row of 3, 1 and 2 rows
def test_any_row_count(M):
    """Token counts that are no multiple of 4 and less than 7/8 of a round of tiles: the two ops
    (whole rounds: test_fused_epilogue_row_counts)."""
    _run_both(M, 512, 4, 128, 90 + M, exact=True)


Q4, H128, H256 = "fp8_gemm_4q<true, 4, 256>", "fp8_gemm_4h<true, 0, 128, 128, 4>", "fp8_gemm_4h<true, 0, 256, 128, 3>"


def _fused_op_kernels(names):
    """The kernels after the two-op sequence's norm/RoPE kernel: the fused op's."""
    i = next((i for i, n in enumerate(names) if n.startswith("qk_norm_rope_kernel")), -1)
    return names[i + 1:]


@pytest.mark.parametrize("M,kernels", [
    (2305, [Q4]), (2306, [Q4]), (2307, [Q4]),  # 10 x 48 tiles: 1, 2 and 3 rows in the last tile row
    (2816, [Q4, H128, "qkv_tail_norm_rope<128>"]), (4353, [Q4, H256, "qkv_tail_norm_rope<256>"]),
    (4355, [Q4, H256, "qkv_tail_norm_rope<256>"]),
    # a short last tile row as quarter tiles beside the leftover ones
    (1560, [Q4, H128, "qkv_tail_norm_rope<128>"]), (1563, [Q4, H128, "qkv_tail_norm_rope<128>"]),
])
@pytest.mark.parametrize("cache_tokens", [-1, 1500])
def test_fused_epilogue_row_counts(M, kernels, cache_tokens):
    """Row counts, odd ones among them, through the fused epilogue and every form of its tail; the ring takes all
    rows or the first 1500."""
    announce("fp8 qkv norm rope row counts", M, cache_tokens)
    _, names = kernels_of(lambda: _run_both(M, 512, 32, 128, M, exact=True, cache_tokens=cache_tokens))
    assert not names or _fused_op_kernels(names) == kernels


# rows below whole rounds, sub-tiles of both kinds, and split-K GEMMs of few tiles (with their workspace)
@pytest.mark.parametrize("M,K,H,fused", [(4100, 1024, 32, True), (4223, 1024, 32, True), (3120, 1024, 32, True),
                                         (1560, 1024, 32, True), (64, 4096, 4, False), (200, 8192, 4, False)])
def test_same_gemm_kernels_as_the_two_ops(M, K, H, fused):
    """Operands whose rounded sums show the order in which a kernel adds them: the op gives every row the GEMM
    kernel that fp8_scaled_mm gives it, so the results are still the two ops' bit for bit."""
    import joyomni_ops as jo
    announce("fp8 qkv norm rope same kernels", M, K, H)
    _, names = kernels_of(lambda: _run_both(M, K, H, 128, M + K, exact="order"))
    assert not names or (Q4 in _fused_op_kernels(names)) == fused
    if M == 4100:  # the operands do show it: 32x32x64 against 16x16x128 MFMAs
        a, b, sa, sw, bias = _problem(M, K, H, 128, M + K, "order")[:5]
        whole = jo.fp8_scaled_mm(a, b, sa, sw, torch.bfloat16, bias)[:600]
        part = jo.fp8_scaled_mm(a[:600], b, sa[:600], sw, torch.bfloat16, bias)
        torch.cuda.synchronize()
        assert 0 < int((whole != part).sum()) < 0.2 * whole.numel()


@pytest.mark.parametrize("outputs", ["ring", "no ring", "q"])
def test_rows_below_whole_rounds_with_fewer_outputs(outputs):
    """4100 tokens: the 4 rows below whole rounds with the ring alone (all of it above them), without ring rows, and
    with Q alone beside the ring."""
    announce("fp8 qkv norm rope rows below whole rounds", outputs)
    kw = {"ring": dict(with_q=False, with_k=False, with_v=False, cache_tokens=4096),
          "no ring": dict(cache_tokens=0), "q": dict(with_k=False, with_v=False, cache_tokens=4098, pre_rope=False)}
    _run_both(4100, 512, 32, 128, 31, exact=True, **kw[outputs])


@pytest.mark.parametrize("with_scratch", [True, False])
def test_less_than_a_round_with_and_without_scratch(with_scratch):
    """1024 rows x 32 heads (192 of 256 tiles) run as the GEMM and the standalone kernel where the scratch is
    given, and in the fused epilogue where it is not: the same bits."""
    announce("fp8 qkv norm rope less than a round", with_scratch)
    import joyomni_ops as jo
    from joyomni_ops import _lib
    M, K, H, D = 1024, 512, 32, 128
    E = H * D
    a, b, sa, sw, bias, qw, kw, cos, sin = _problem(M, K, H, D, 77, True)
    need = jo._LIB.joy_fp8_qkv_norm_rope_cache_scratch_size(M, K, H, D)
    assert need == M * 3 * E * 2
    ref = _outputs(M, H, D, 1, M, 78)
    got = tuple(t.clone() for t in ref)
    y = jo.fp8_scaled_mm(a, b, sa, sw, torch.bfloat16, bias)
    jo.fused_qkv_norm_rope_cache(y, H, 1e-6, qw, kw, cos, sin, ref[0], ref[1], ref[3], ref[4], 0, 0, v_out=ref[2])
    scratch = torch.empty(need if with_scratch else 16, dtype=torch.uint8, device=DEV)
    _lib.check(jo._LIB, jo._LIB.joy_fp8_qkv_norm_rope_cache(
        a.data_ptr(), b.data_ptr(), sa.data_ptr(), sw.data_ptr(), bias.data_ptr(), M, K, H, D, 1e-6, qw.data_ptr(),
        kw.data_ptr(), cos.data_ptr(), sin.data_ptr(), got[0].data_ptr(), E, got[1].data_ptr(), E, got[2].data_ptr(), E,
        got[3].data_ptr(), got[4].data_ptr(), 1, M, 0, 0, M, 0, scratch.data_ptr(), scratch.numel(),
        torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    for name, r, o in zip(("q_out", "k_out", "v_out", "ring K", "ring V"), ref, got):
        assert torch.equal(u16_t(r), u16_t(o)), name


@pytest.mark.parametrize("M", [1, 3, 1028])  # 192 tiles; five rows of 192 tiles, with 4 rows below whole rounds
@pytest.mark.parametrize("with_scratch", [True, False])
def test_many_heads_with_and_without_scratch(M, with_scratch):
    """128 heads: shapes whose tiles could all take the fused epilogue run without any scratch, also where the scratch
    would send them, or the rows below whole rounds, through the GEMM and the standalone kernel."""
    announce("fp8 qkv norm rope many heads", M, with_scratch)
    import joyomni_ops as jo
    from joyomni_ops import _lib
    K, H, D = 512, 128, 128
    E = H * D
    a, b, sa, sw, bias, qw, kw, cos, sin = _problem(M, K, H, D, 7 + M, True)
    need = jo._LIB.joy_fp8_qkv_norm_rope_cache_scratch_size(M, K, H, D)
    if M < 4 and not with_scratch:
        assert need >= M * 3 * E * 2
        return  # fewer than 4 rows do not take the epilogue
    ref = _outputs(M, H, D, 1, M, 8)
    got = tuple(t.clone() for t in ref)
    y = jo.fp8_scaled_mm(a, b, sa, sw, torch.bfloat16, bias)
    jo.fused_qkv_norm_rope_cache(y, H, 1e-6, qw, kw, cos, sin, ref[0], ref[1], ref[3], ref[4], 0, 0, v_out=ref[2])
    scratch = torch.empty(max(need, 16) if with_scratch else 16, dtype=torch.uint8, device=DEV)
    call = lambda: _lib.check(jo._LIB, jo._LIB.joy_fp8_qkv_norm_rope_cache(  # noqa: E731
        a.data_ptr(), b.data_ptr(), sa.data_ptr(), sw.data_ptr(), bias.data_ptr(), M, K, H, D, 1e-6, qw.data_ptr(),
        kw.data_ptr(), cos.data_ptr(), sin.data_ptr(), got[0].data_ptr(), E, got[1].data_ptr(), E, got[2].data_ptr(), E,
        got[3].data_ptr(), got[4].data_ptr(), 1, M, 0, 0, M, 0, scratch.data_ptr() if with_scratch else None,
        scratch.numel() if with_scratch else 0, torch.cuda.current_stream().cuda_stream))
    _, names = kernels_of(call)
    assert not names or (names == [Q4]) == (not with_scratch)
    for name, r, o in zip(("q_out", "k_out", "v_out", "ring K", "ring V"), ref, got):
        assert torch.equal(u16_t(r), u16_t(o)), name
