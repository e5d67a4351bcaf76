"""GPU parity: joint-attention core (joyomni_ops.sdpa_attention, joy_attention_fwd) vs the
float64 oracle (oracle/attention.py, restating dit.py:154-167).

Tolerance (bf16 output, probabilities rounded to bf16 for the P V product as in bf16
flash attention): |out - ref| <= 2^-8 * (max_j |v[j, h, :]| + |ref|) per element. Exact
cases (single key, identical keys over small-integer values) are checked bit for bit."""
import math

import numpy as np
import pytest
import torch

from gpu_util import DEV, announce, gen, u16
from oracle import attention as oa
from oracle.fp8 import bf16_to_f32, f32_to_bf16

pytestmark = pytest.mark.gpu


def _inputs(Lq, Lk, H, seed, scale=1.0):
    g = gen(seed)
    q = (torch.randn(Lq, H, 128, generator=g) * scale).to(torch.bfloat16)
    k = (torch.randn(Lk, H, 128, generator=g) * scale).to(torch.bfloat16)
    v = torch.randn(Lk, H, 128, generator=g).to(torch.bfloat16)
    return q, k, v


def _run(q, k, v, scale=None):
    import joyomni_ops as jo
    out = jo.sdpa_attention(q[None].to(DEV), k[None].to(DEV), v[None].to(DEV), scale)
    torch.cuda.synchronize()
    return out[0]


def _check(out, q, k, v, what, scale=None, rows=None):
    ref = oa.sdpa(u16(q if rows is None else q[rows]), u16(k), u16(v), scale)
    got = bf16_to_f32(u16(out if rows is None else out[torch.from_numpy(rows).to(out.device)]))
    vmax = np.abs(bf16_to_f32(u16(v))).max(axis=0)  # [H, D] -> per head max below
    tol = 2.0 ** -8 * (vmax.max(axis=-1)[None, :, None] + np.abs(ref))
    err = np.abs(got - ref)
    assert (err <= tol).all(), f"{what}: {np.count_nonzero(err > tol)} elements beyond tolerance, max err {err.max():.3e}"
    return err.max()


@pytest.mark.parametrize("Lq,Lk,H", [(1, 1, 1), (5, 3, 2), (128, 64, 1), (130, 65, 2), (300, 700, 3),
                                     (257, 129, 4), (64, 1000, 1), (33, 32, 2), (40, 33, 1), (70, 96, 2)])
def test_random_shapes(Lq, Lk, H):
    announce("attention random", Lq, Lk, H)
    q, k, v = _inputs(Lq, Lk, H, Lq * 31 + Lk)
    _check(_run(q, k, v), q, k, v, f"{Lq}x{Lk}x{H}")


@pytest.mark.parametrize("Lq,H", [(330, 7), (256, 3), (225, 2), (40, 9)])
def test_workgroups_straddling_heads(Lq, H):
    """Workgroups take 8 consecutive 32-query blocks of the head-major block list, so one
    workgroup can hold the end of one head and the start of the next (330 queries: 11 blocks per
    head), or padding blocks past Lq (40 queries: 2 of 8 blocks); every row of every head is
    checked."""
    announce("attention straddling heads", Lq, H)
    q, k, v = _inputs(Lq, 300, H, Lq + 17 * H)
    _check(_run(q, k, v), q, k, v, f"{Lq}x300x{H}")


def test_peaked_scores_and_explicit_scale():
    """Large-magnitude q/k (peaked softmax, exp2 range) and a non-default scale."""
    announce("attention peaked")
    q, k, v = _inputs(200, 333, 2, 7, scale=3.0)
    _check(_run(q, k, v), q, k, v, "peaked")
    _check(_run(q, k, v, 0.02), q, k, v, "scale 0.02", scale=0.02)


def test_running_max_jumps_across_tiles():
    """Scores that jump between 64-key tiles, so that the softmax's first pass against the running
    max fails its check and the max-based pass takes over in every way it can: a jump of about 5
    and 7.9 (log2 units, below the slack of 8: the sum check fails, the running max stays), of
    about 12.7 (the running max moves and O is rescaled), a drop of about 20 (tiny probabilities,
    the first pass holds) and of about 200 (probabilities against the old max overflow to inf).
    Key rows carry their level in dimension 0 and queries 4 there, on top of small random parts;
    the last tile is partial (17 keys)."""
    announce("attention running-max jumps")
    g = gen(41)
    Lq, H, tiles = 96, 2, 11
    Lk = 64 * (tiles - 1) + 17
    q = torch.randn(Lq, H, 128, generator=g) * 0.1
    k = torch.randn(Lk, H, 128, generator=g) * 0.1
    v = torch.randn(Lk, H, 128, generator=g)
    q[:, :, 0] = 4.0
    # level of dimension 0 per tile: scores move by 4 * level / sqrt(128) * log2(e) ~ 0.51 * level
    levels = {0: 0.0, 3: 10.0, 4: 15.5, 6: 25.0, 7: -40.0, 8: 400.0, 9: 0.0, 10: 401.0}
    for t, lv in levels.items():
        rows = slice(64 * t, min(64 * (t + 1), Lk))
        k[rows, 0, 0] = lv
        k[rows, 1, 0] = -lv if t in (3, 7) else lv  # head 1: drops where head 0 jumps
    q, k, v = q.to(torch.bfloat16), k.to(torch.bfloat16), v.to(torch.bfloat16)
    out = _run(q, k, v)
    assert torch.isfinite(out.float()).all()
    _check(out, q, k, v, "running-max jumps")


def test_single_key_is_exact():
    announce("attention single key")
    q, k, v = _inputs(77, 1, 3, 11)
    assert np.array_equal(u16(_run(q, k, v)), np.broadcast_to(u16(v), (77, 3, 128)))


@pytest.mark.parametrize("Lk", [64, 40])
def test_identical_keys_exact_mean(Lk):
    """Lk identical keys (a full tile; a tile whose second 32-key half is partly past the end):
    every probability is exactly 1, small-integer values sum exactly, so the output is the bf16
    rounding of their mean."""
    announce("attention identical keys", Lk)
    rng = np.random.default_rng(5)
    H = 2
    q = torch.from_numpy(rng.standard_normal((40, H, 128)).astype(np.float32)).to(torch.bfloat16)
    k = torch.from_numpy(np.repeat(rng.standard_normal((1, H, 128)).astype(np.float32), Lk, axis=0)
                         ).to(torch.bfloat16)
    v = torch.from_numpy(rng.integers(-8, 9, (Lk, H, 128)).astype(np.float32)).to(torch.bfloat16)
    exp = f32_to_bf16((bf16_to_f32(u16(v)).astype(np.float64).mean(axis=0)).astype(np.float32))
    assert np.array_equal(u16(_run(q, k, v)), np.broadcast_to(exp, (40, H, 128)))


def test_strided_views_and_out_rows():
    """q/k/v read as head/token-strided slices of fused [L, 3, H, D] rows; output written into
    the rows of a wider [L, H*D + 64] buffer (only the [:, :H*D] part may change)."""
    announce("attention strided")
    import joyomni_ops as jo
    L, H = 190, 2
    g = gen(3)
    qkv = torch.randn(L, 3, H, 128, generator=g).to(torch.bfloat16).to(DEV)
    q, k, v = qkv[None, :, 0], qkv[None, :, 1], qkv[None, :, 2]
    buf = torch.full((L, H * 128 + 64), 7.0, dtype=torch.bfloat16, device=DEV)
    out = buf[:, :H * 128].view(1, L, H, 128)
    jo.sdpa_attention_out(q, k, v, out)
    torch.cuda.synchronize()
    assert bool((buf[:, H * 128:] == 7.0).all())
    _check(out[0], q[0].cpu(), k[0].cpu(), v[0].cpu(), "strided")


def test_batch_of_two():
    announce("attention batch 2")
    import joyomni_ops as jo
    g = gen(4)
    q = torch.randn(2, 70, 2, 128, generator=g).to(torch.bfloat16)
    k = torch.randn(2, 90, 2, 128, generator=g).to(torch.bfloat16)
    v = torch.randn(2, 90, 2, 128, generator=g).to(torch.bfloat16)
    out = jo.sdpa_attention(q.to(DEV), k.to(DEV), v.to(DEV))
    torch.cuda.synchronize()
    for b in range(2):
        _check(out[b], q[b], k[b], v[b], f"batch {b}")


def test_argument_errors():
    import joyomni_ops as jo
    q = torch.zeros(1, 4, 2, 64, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(RuntimeError, match="head_dim=128"):
        jo.sdpa_attention(q, q, q)
    q = torch.zeros(1, 4, 2, 128, dtype=torch.bfloat16, device=DEV)
    k = torch.zeros(1, 0, 2, 128, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(RuntimeError, match="empty key"):
        jo.sdpa_attention(q, k, k)


def test_cfg4_joint_shape_sampled_queries():
    """The block's joint attention: 10800 + 512 queries over 2 x 10800 cached + 10800 + 512 keys,
    40 heads. 64 sampled queries (queries are independent) against the oracle; torch's SDPA
    (the reference's own call) on the same inputs is held to the same tolerance."""
    announce("attention cfg4 11312 x 32912 x 40")
    Lq, Lk, H = 11312, 32912, 40
    q, k, v = _inputs(Lq, Lk, H, 2024)
    qd, kd, vd = q[None].to(DEV), k[None].to(DEV), v[None].to(DEV)
    import joyomni_ops as jo
    out = jo.sdpa_attention(qd, kd, vd)[0]
    ref_sdpa = torch.nn.functional.scaled_dot_product_attention(
        qd.transpose(1, 2), kd.transpose(1, 2), vd.transpose(1, 2), is_causal=False).transpose(1, 2)[0]
    torch.cuda.synchronize()
    rows = np.sort(np.random.default_rng(9).choice(Lq, 64, replace=False))
    rows[-1] = Lq - 1
    err_ours = _check(out, q, k, v, "cfg4 ours", rows=rows)
    err_sdpa = _check(ref_sdpa, q, k, v, "cfg4 torch sdpa", rows=rows)
    print(f"cfg4 max|err| vs float64: ours {err_ours:.3e}, torch SDPA {err_sdpa:.3e}")


@pytest.mark.parametrize("Lk", [3467, 11267])
def test_reference_production_shape_sampled_queries(Lk):
    """The reference's own production attention (480x832 chunk: 3467 queries over 3467..11267
    keys, 32 heads of 128): 48 sampled queries against the oracle. 3467 = 108 blocks of 32 + 11
    rows: a partial last query block, 108 blocks per head (workgroups straddle heads), and a
    partial last key tile (11267 = 176 tiles of 64 + 3 keys)."""
    announce("attention reference production", 3467, Lk, 32)
    Lq, H = 3467, 32
    q, k, v = _inputs(Lq, Lk, H, 77 + Lk)
    out = _run(q, k, v)
    rows = np.sort(np.random.default_rng(Lk).choice(Lq, 48, replace=False))
    rows[0], rows[-1] = 0, Lq - 1
    _check(out, q, k, v, f"production {Lq}x{Lk}x{H}", rows=rows)


def _split_call(q, k, v, workspace):
    """joy_attention_fwd_workspace on [L, H, 128] device tensors, with its workspace or with none."""
    import ctypes
    import joyomni_ops as jo
    from joyomni_ops import _lib
    lib, H = jo._LIB, q.size(1)
    view = lambda t: ctypes.byref(_lib.Bf16View(t.data_ptr(), t.size(0), t.stride(0), t.stride(1)))  # noqa: E731
    nbytes = lib.joy_attention_workspace_size(q.size(0), k.size(0), H) if workspace else 0
    ws = torch.full((nbytes + 64,), 0xff, dtype=torch.uint8, device=DEV)  # NaN where nothing is written
    out = torch.full_like(q, float("nan"))
    st = lib.joy_attention_fwd_workspace(view(q), view(k), view(v), out.data_ptr(), H * 128, H, 128,
                                         1 / math.sqrt(128), ws.data_ptr(), nbytes,
                                         torch.cuda.current_stream().cuda_stream)
    _lib.check(lib, st)
    torch.cuda.synchronize()
    assert bool((ws[nbytes:] == 0xff).all())
    return nbytes, out


# few groups with many parts; parts and a shorter last one; a whole round before the split groups (257 and 264
# groups on 256 CUs); a partial key tile alone in the last part, and none; padding blocks in the last group
@pytest.mark.parametrize("Lq,Lk,H", [(1, 4001, 1), (100, 1600, 3), (512, 1025, 32), (859, 2001, 32), (65, 1152, 40),
                                     (2056, 1400, 32), (2100, 2100, 32), (330, 3000, 7)])
def test_key_split_matches_unsplit_and_oracle(Lq, Lk, H):
    """The key split against the unsplit call: both round the probabilities to bf16 against their own
    running max (2^-9 of a weight each) and the result to bf16 (2^-9), so each element is within 2^-7 of
    max|v| + |ref| of the other; sampled rows against the oracle as everywhere."""
    announce("attention key split", Lq, Lk, H)
    q, k, v = _inputs(Lq, Lk, H, Lq * 7 + Lk)
    qd, kd, vd = q.to(DEV), k.to(DEV), v.to(DEV)
    none, whole = _split_call(qd, kd, vd, False)
    nbytes, split = _split_call(qd, kd, vd, True)
    assert none == 0 and nbytes > 0
    vmax = vd.float().abs().amax(dim=(0, 2))[None, :, None]
    assert bool(((split.float() - whole.float()).abs() <= 2.0 ** -7 * (vmax + whole.float().abs())).all())
    rows = np.unique(np.random.default_rng(Lk).choice(Lq, min(Lq, 24)))
    rows[-1] = Lq - 1
    _check(split, q, k, v, f"split {Lq}x{Lk}x{H}", rows=rows)


def test_key_split_with_parts_that_add_nothing():
    """Keys of whole parts with scores of -inf (an infinite key component against positive queries) and
    rising scores from part to part: the -inf keys weigh nothing, wherever the parts begin."""
    announce("attention key split -inf")
    Lq, Lk, H = 64, 2048, 4
    q, k, v = _inputs(Lq, Lk, H, 5)
    q[:, :, 0] = q[:, :, 0].abs() + 0.5
    k[:, :, 1] = (torch.arange(Lk) / 64)[:, None].to(torch.bfloat16)
    k[: Lk // 4, :, 0] = float("-inf")
    k[Lk // 2: Lk // 2 + 300, :, 0] = float("-inf")
    nbytes, out = _split_call(q.to(DEV), k.to(DEV), v.to(DEV), True)
    assert nbytes > 0
    keep = torch.isfinite(k[:, 0, 0])
    _check(out, q, k[keep], v[keep], "split -inf")


@pytest.mark.parametrize("Lq,Lk,H", [(40, 100, 1), (64, 2048, 4)])  # unsplit; parts along the keys
def test_scores_near_the_lowest_float(Lq, Lk, H):
    """Finite scores close to the lowest float (masks written into the keys) are scores like others: the
    highest of them take the whole weight, here every third key at -3.2e38 in units of log2 against -3.3e38."""
    announce("attention lowest scores", Lq, Lk, H)
    import joyomni_ops as jo
    assert (jo._LIB.joy_attention_workspace_size(Lq, Lk, H) > 0) == (Lk == 2048)
    q, k, v = _inputs(Lq, Lk, H, 21)
    q.zero_()[:, :, 0] = 1
    k[:, :, 0] = -3.3e38
    k[1::3, :, 0] = -3.2e38
    _check(_run(q, k, v, math.log(2)), q, k, v, "lowest scores", scale=math.log(2))


def test_key_split_in_a_captured_graph():
    """sdpa_attention with a split captured into a HIP graph and replayed with eager work between."""
    announce("attention key split captured")
    import joyomni_ops as jo
    q, k, v = (t[None].to(DEV) for t in _inputs(512, 2000, 16, 6))
    ref = jo.sdpa_attention(q, k, v)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            out = jo.sdpa_attention(q, k, v)
    for _ in range(3):
        out.fill_(float("nan"))
        jo.sdpa_attention(q.flip(1), v, k)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref)


@pytest.mark.parametrize("through", ["wrapper", "torch.ops"])
def test_c_abi_refusals_are_joy_errors(through):
    """What the C ABI refuses under an operator is raised as the package's JoyError, with its text; an operator's own
    argument check as a RuntimeError that is none."""
    announce("JoyError", through)
    import joyomni_ops as jo
    from joyomni_ops import _lib
    op = jo.sdpa_attention if through == "wrapper" else torch.ops.joyomni_ops.sdpa_attention
    x = torch.zeros(1, 4, 2, 64, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(_lib.JoyError, match="head_dim=128 only"):
        op(x, x, x)
    with pytest.raises(RuntimeError, match="same shape") as e:
        op(x, x, x[:, :2])
    assert not isinstance(e.value, _lib.JoyError)
    y = torch.zeros(1, 4, 2, 128, dtype=torch.bfloat16, device=DEV)
    assert not op(y, y, y).any()  # and the next call is an ordinary one
