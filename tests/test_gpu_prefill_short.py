"""GPU parity of prefill_small_kernel beyond the shapes of test_gpu_prefill.py, which forces the 128-wide kernel's shapes in turn: here the
library chooses."""
import ctypes as C

import pytest
import torch

from oracle import attn_oracle as orc
from tests.helpers import assert_inplace_o_close, assert_lse_close, assert_o_close, meta, rand_t

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _dev(*ts):
    return [t.to(DEV) for t in ts]


@pytest.mark.parametrize("mode", ["partial", "accumulate", "in_place"])
@pytest.mark.parametrize("D,dtype", [(128, torch.float16), (128, torch.bfloat16), (64, torch.float16), (16, torch.bfloat16)])
def test_nan_scores_reach_the_rows_that_see_them(lsa, mode, D, dtype):
    """A NaN in a K row and in a Q row (short prompts of 128-wide heads, small heads): the rows that meet one become NaN, outputs and
    running state, stay NaN through a second step, and no other row changes by more than its rounding."""
    print("case", mode, D, dtype, flush=True)
    lens, Hq, Hkv = [100, 33], 4, 2
    T = sum(lens)
    q, k, v = rand_t((T, Hq, D), 81, dtype), rand_t((T, Hkv, D), 82, dtype), rand_t((T, Hkv, D), 83, dtype)
    m = meta(lens)
    o_ref, lse_ref = orc.attn_step(q, k, v, *m, *m, 1)
    qn, kn = q.clone(), k.clone()
    kn[10, 0, 3] = float("nan")   # key 10 of the first request, heads 0 and 1
    qn[105, 2, 0] = float("nan")  # row 5 of the second request, head 2
    hit = torch.zeros((T, Hq), dtype=torch.bool)
    hit[10:100, :2] = True
    hit[105, 2] = True
    qd, kd, vd, md = *_dev(qn, kn, v), _dev(*m)
    if mode == "in_place":
        o = torch.full((T, Hq, D), 7.0, dtype=dtype, device=DEV)
        ms, ls = torch.full((T, Hq), float("-inf"), device=DEV), torch.zeros((T, Hq), device=DEV)
        step = lambda K: lsa.context_attention_fwd(qd, K, vd, o, *md, *md, 1, max(lens), ms, ls, total_q_len=T)
        lse_of = lambda: orc.state_lse(ms.cpu(), ls.cpu()).float()
    else:
        o, lse = torch.full((T, Hq, D), 7.0, device=DEV), torch.full((T, Hq), float("-inf"), device=DEV)
        step = lambda K: lsa.prefill_attention_step(qd, K, vd, *md, *md, 1, max(lens), o, lse, accumulate=mode == "accumulate", total_q_len=T)
        lse_of = lambda: lse.cpu()
    step(kd)
    torch.cuda.synchronize()
    got, got_lse = o.float().cpu(), lse_of()
    assert torch.equal(got.isnan().all(-1), hit) and torch.equal(got.isnan().any(-1), hit) and torch.equal(got_lse.isnan(), hit)
    got[hit], got_lse[hit] = o_ref.float()[hit], lse_ref.float()[hit]
    if mode == "in_place":
        assert_inplace_o_close(got.to(dtype), o_ref.to(dtype), o_ref, "o")
    else:
        assert_o_close(got, o_ref, "O")
    assert_lse_close(got_lse, lse_ref, "LSE")
    if mode != "partial":  # the same keys once more, without the NaN in K: the rows stay NaN
        step(k.to(DEV))
        torch.cuda.synchronize()
        assert torch.equal(o.float().cpu().isnan().all(-1), hit) and torch.equal(lse_of().isnan(), hit)


@pytest.mark.parametrize("rows", [100, 2000])
def test_v_f16_valid_needs_the_copy_whatever_kernel_runs(lsa, rows):
    """Short prompts (whose kernel converts a bfloat16 V itself) and longer ones: the flag without the buffer, or with one that cannot be
    the copy, is refused by both operators."""
    q, k, v = (torch.zeros((rows, 2, 128), dtype=torch.bfloat16, device=DEV) for _ in range(3))
    md = _dev(*meta([rows]))
    o, m, l = torch.zeros_like(q), torch.zeros((rows, 2), device=DEV), torch.zeros((rows, 2), device=DEV)
    for held in (None, v, torch.zeros((rows, 1, 128), dtype=torch.float16, device=DEV)):
        with pytest.raises(ValueError, match="v_f16_valid needs v_f16"):
            lsa.prefill_attention_step(q, k, v, *md, *md, 1, rows, v_f16=held, v_f16_valid=True)
        with pytest.raises(ValueError, match="v_f16_valid needs v_f16"):
            lsa.context_attention_fwd(q, k, v, o, *md, *md, 1, rows, m, l, v_f16=held, v_f16_valid=True)
    for t in (q, k, v):
        t.normal_().mul_(8).round_().div_(8)  # (exact in fp16 too)
    want = lsa.prefill_attention_step(q, k, v, *md, *md, 1, rows)
    got = lsa.prefill_attention_step(q, k, v, *md, *md, 1, rows, v_f16=v.half(), v_f16_valid=True)
    torch.cuda.synchronize()
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_short_rows_behind_one_long_context_and_bounded_ones(lsa, dtype):
    """A batch of short chunks of which one has a long context (the 128-wide kernel) and one whose contexts the caller bounds (the
    kernel of short prompts), through the native pass and the checked one."""
    for lens, ctx, bound in [([64, 33, 64, 1], [0, 2500, 0, 7], None), ([64, 33, 64, 1], [700, 900, 0, 960], 961)]:
        klens = [n + c for n, c in zip(lens, ctx)]
        T = sum(lens)
        q, kv = rand_t((T, 8, 128), 91, dtype), rand_t((sum(klens), 4, 128), 92, dtype)
        qm, km = meta(lens, ctx), meta(klens)
        o_ref, lse_ref = orc.attn_step(q, kv[:, :2].contiguous(), kv[:, 2:].contiguous(), *qm, *km, 1)
        qd, kvd = q.to(DEV), kv.to(DEV)
        k, v = kvd[:, :2], kvd[:, 2:]
        for given in (bound, None if bound is None else torch.tensor(bound)):  # (a tensor goes through the checked pass)
            o, lse = lsa.prefill_attention_step(qd, k, v, *_dev(*qm), *_dev(*km), 1, max(lens), total_q_len=T, max_kv_len=given)
            torch.cuda.synchronize()
            assert_o_close(o, o_ref, "O")
            assert_lse_close(lse, lse_ref, "LSE")


SMALL_16, SMALL_32, SMALL_TURNS = 1, 2, 3  # LSATTN_ROUTE_* of include/lsattn.h


def _every_epilogue_on(route, lsa, mode, V, D, Hq, Hkv, lens, ctx, spare=0):
    """One step (the partial) or two over halves of the keys (the folding epilogues) against the oracle, each of them on `route`.
    V: "f16", "bf16" (converted by the kernel) or "bf16 copied" (the caller's buffer for the fp16 copy).  spare: rows of the K/V
    buffers behind the last request's."""
    from loongserve_amd import _lib, ops
    dtype = torch.float16 if V == "f16" else torch.bfloat16
    klens = [n + c for n, c in zip(lens, ctx)]
    T, TK = sum(lens), sum(klens)
    q, k, v = rand_t((T, Hq, D), 71, dtype), rand_t((TK, Hkv, D), 72, dtype), rand_t((TK, Hkv, D), 73, dtype)
    ramp = torch.cat([torch.arange(n) % 400 for n in klens]).float() / 80 + 1  # (the running maxima are raised again and again)
    k = (k.float() * ramp[:, None, None]).to(dtype)
    qm, km = meta(lens, ctx), meta(klens)
    o_ref, lse_ref = orc.attn_step(q, k, v, *qm, *km, 1)
    half = [n // 2 for n in klens]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32)
    steps = [(km[0], i32(half), i32([0] * len(lens))), (km[0] + i32(half), i32([n - f for n, f in zip(klens, half)]), i32(half))]
    qd, kd, vd, qmd = *_dev(q, k, v), _dev(*qm)
    if spare:
        kd, vd = (torch.cat([x, x.new_full((spare, Hkv, D), float("nan"))]) for x in (kd, vd))
    kw = dict(v_f16=torch.empty(vd.shape, dtype=torch.float16, device=DEV)) if V == "bf16 copied" else {}

    def on_route(o, s):
        a = ops._prefill_args(qd, kd, vd, o, *qmd, *s, 1, max(lens), None, total_q_len=T, **kw)
        assert _lib.load().lsattn_prefill_route(C.byref(a)) == route and a.v_is_f16 == (V == "bf16 copied")
        return s

    if mode == "in_place":
        o = torch.full((T, Hq, D), 7.0, dtype=dtype, device=DEV)
        m, l = torch.full((T, Hq), float("-inf"), device=DEV), torch.zeros((T, Hq), device=DEV)
        o_st, m_st, l_st = torch.zeros((T, Hq, D), dtype=dtype), torch.full((T, Hq), float("-inf")), torch.zeros(T, Hq)
        for s in steps:
            lsa.context_attention_fwd(qd, kd, vd, o, *qmd, *on_route(o, _dev(*s)), 1, max(lens), m, l, total_q_len=T, **kw)
            orc.context_attention_fwd(q, k, v, o_st, *qm, *s, 1, max(lens), m_st, l_st)
        torch.cuda.synchronize()
        assert_inplace_o_close(o.cpu(), o_st, o_ref, "o")
        assert_lse_close(orc.state_lse(m.cpu(), l.cpu()).float(), lse_ref, "state LSE")
        return
    o, lse = torch.full((T, Hq, D), 7.0, device=DEV), torch.full((T, Hq), float("-inf"), device=DEV)
    for s in steps if mode == "accumulate" else [km]:
        lsa.prefill_attention_step(qd, kd, vd, *qmd, *on_route(o, _dev(*s)), 1, max(lens), o, lse, accumulate=mode == "accumulate",
                                   total_q_len=T, **kw)
    torch.cuda.synchronize()
    assert_o_close(o, o_ref, "O")
    assert_lse_close(lse, lse_ref, "LSE")


@pytest.mark.parametrize("mode", ["partial", "accumulate", "in_place"])
@pytest.mark.parametrize("V", ["f16", "bf16", "bf16 copied"])
@pytest.mark.parametrize("Hq,Hkv", [(32, 32), (16, 8), (16, 4)])
def test_short_prompts_with_32_positions_per_wave(lsa, mode, V, Hq, Hkv):
    """128-wide heads, more workgroups than the 16-position shape takes: one, two and four heads side by side, prompts around the waves'
    32 rows and the 64-key tiles, some behind a context."""
    print("case", mode, V, Hq, Hkv, flush=True)
    _every_epilogue_on(SMALL_32, lsa, mode, V, 128, Hq, Hkv, [128, 100, 7, 256, 65, 33] * 4, [0, 40] * 12)


@pytest.mark.parametrize("mode", ["partial", "accumulate", "in_place"])
@pytest.mark.parametrize("V", ["f16", "bf16", "bf16 copied"])
@pytest.mark.parametrize("D", [64, 32, 16])
def test_requests_that_take_turns_in_the_grid(lsa, mode, V, D):
    """Heads of 16 to 64 in a ragged batch whose places in the grid turn from tile to tile."""
    print("case", mode, V, D, flush=True)
    _every_epilogue_on(SMALL_TURNS, lsa, mode, V, D, 16, 4, [1500, 1200, 1, 33, 1000, 64, 1301, 900], [0] * 8)


@pytest.mark.parametrize("mode", ["partial", "accumulate", "in_place"])
@pytest.mark.parametrize("V", ["f16", "bf16", "bf16 copied"])
@pytest.mark.parametrize("what", ["stages", "turns", "bunches", "bunches of 64", "bunches by K/V"])
def test_short_prompts_in_three_stages_and_the_grids_orders(lsa, mode, V, what):
    """128-wide heads with 32 positions per wave: prompts around multiples of the 32-key tiles and their three stages; a ragged batch whose
    requests take turns; and grids that take a few requests at a time, by the count of workgroups (a last bunch that is short) and,
    where the K/V that the requests read is larger than the L2s, by that."""
    print("case", mode, V, what, flush=True)
    if what == "stages":
        _every_epilogue_on(SMALL_32, lsa, mode, V, 128, 16, 4, [31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128, 129, 159, 161, 191, 193] * 2, [0, 31, 1, 0] * 8)
    elif what == "turns":
        _every_epilogue_on(SMALL_TURNS, lsa, mode, V, 128, 32, 8, [700, 300, 650, 1], [0] * 4)
    elif what == "bunches":
        _every_epilogue_on(SMALL_32, lsa, mode, V, 128, 16, 8, [130] * 19 + [97], [0] * 20)
    elif what == "bunches of 64":
        _every_epilogue_on(SMALL_32, lsa, mode, V, 64, 16, 16, [130] * 72 + [1], [0] * 73)
    else:
        _every_epilogue_on(SMALL_32, lsa, mode, V, 128, 32, 32, [700, 33, 650, 64, 1, 600, 400, 20, 768, 512, 129, 300, 300], [0] * 13, spare=64)


@pytest.mark.parametrize("mode", ["partial", "accumulate", "in_place"])
@pytest.mark.parametrize("V", ["f16", "bf16", "bf16 copied"])
@pytest.mark.parametrize("Hq,Hkv,lens", [(20, 20, [1024, 993]), (8, 2, [897, 30, 800])])
def test_longer_prompts_with_16_positions_per_wave(lsa, mode, V, Hq, Hkv, lens):
    print("case", mode, V, Hq, Hkv, flush=True)
    _every_epilogue_on(SMALL_16, lsa, mode, V, 128, Hq, Hkv, lens, [0] * len(lens))


@pytest.mark.parametrize("Hq,Hkv", [(8, 1), (24, 24)])
def test_lone_prompts_past_1280_rows(lsa, Hq, Hkv):
    """The longest prompt that the kernel folds in place.  (The route that is asked for names no m: it is the 128-row one of the partial.)"""
    print("case", Hq, Hkv, flush=True)
    _every_epilogue_on(5, lsa, "in_place", "f16", 128, Hq, Hkv, [1472], [0])


@pytest.mark.parametrize("mode", ["partial", "accumulate", "in_place"])
@pytest.mark.parametrize("V", ["f16", "bf16", "bf16 copied"])
@pytest.mark.parametrize("Hq,Hkv,lens,ctx", [(8, 2, [545, 33, 512], [0, 0, 0]), (8, 1, [640, 1, 31], [0, 300, 0]), (20, 20, [768], [0]), (6, 3, [577, 64], [33, 100])])
def test_two_waves_that_share_a_tile(lsa, mode, V, Hq, Hkv, lens, ctx):
    """Up to a workgroup of 64 rows per CU from 512 keys on: one, two and four heads side by side, waves that see one part of a tile or none."""
    print("case", mode, V, Hq, Hkv, lens, flush=True)
    _every_epilogue_on(SMALL_16, lsa, mode, V, 128, Hq, Hkv, lens, ctx)


@pytest.mark.parametrize("V", ["f16", "bf16 copied"])
@pytest.mark.parametrize("Hq,Hkv,n,ctx", [(8, 1, 2048, 0), (4, 4, 1025, 0), (32, 8, 200, 1848), (12, 4, 77, 1300)])
def test_lone_requests_whose_tiles_two_waves_share(lsa, V, Hq, Hkv, n, ctx):
    """One request folded in place, past what other steps bring to the kernel (the route asked for here names no m: it is the 128-wide kernel's)."""
    print("case", V, Hq, Hkv, n, ctx, flush=True)
    _every_epilogue_on(SMALL_16 if n == 1025 and V == "f16" else 5, lsa, "in_place", V, 128, Hq, Hkv, [n], [ctx])


@pytest.mark.parametrize("Hq,Hkv,lens", [(8, 8, [801] * 10), (8, 1, [1280] * 9), (18, 6, [1024] * 4)])
def test_equal_prompts_in_place_with_a_third_workgroup_per_cu(lsa, Hq, Hkv, lens):
    """Between two and three workgroups of 32 positions per CU (the route asked for here names no m: it is the 128-wide kernel's)."""
    print("case", Hq, Hkv, lens, flush=True)
    _every_epilogue_on(4, lsa, "in_place", "f16", 128, Hq, Hkv, lens, [0] * len(lens))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("key", [0, 31, 40, 575])
def test_nan_keys_in_either_part_of_a_tile(lsa, dtype, key):
    """A NaN in one K row of a prompt whose tiles two waves share: the rows that see it become NaN, the others stay."""
    print("case", dtype, key, flush=True)
    n, Hq, Hkv = 600, 8, 2
    q, k, v = _dev(*(rand_t((n, h, 128), 91 + i, dtype) for i, h in enumerate((Hq, Hkv, Hkv))))
    md = _dev(*meta([n]))
    want, want_lse = lsa.prefill_attention_step(q, k, v, *md, *md, 1, n, total_q_len=n)
    k[key, 1, 5] = float("nan")
    got, lse = lsa.prefill_attention_step(q, k, v, *md, *md, 1, n, total_q_len=n)
    hit = torch.zeros((n, Hq), dtype=torch.bool, device=DEV)
    hit[key:, Hq // 2:] = True
    assert torch.equal(got.isnan().all(-1), hit) and torch.equal(got.isnan().any(-1), hit) and torch.equal(lse.isnan(), hit)
    # (a NaN makes a wave raise all its maxima, which moves its other rows by the rounding of their weights to fp16)
    assert_o_close(got[~hit].cpu(), want[~hit].cpu(), "O")
    assert_lse_close(lse[~hit].cpu(), want_lse[~hit].cpu(), "LSE")


@pytest.mark.parametrize("mode", ["partial", "accumulate", "in_place"])
@pytest.mark.parametrize("V", ["f16", "bf16", "bf16 copied"])
@pytest.mark.parametrize("Hq,Hkv,lens,ctx", [(8, 2, [449, 33, 448], [0, 0, 0]), (4, 1, [50, 1], [0, 600]), (32, 16, [1000, 650], [0, 0]), (20, 20, [1153, 1], [0, 0])])
def test_two_waves_that_share_a_tile_of_64_wide_heads(lsa, mode, V, Hq, Hkv, lens, ctx):
    """One, two and three workgroups per CU, one, two and four heads side by side."""
    print("case", mode, V, Hq, Hkv, lens, flush=True)
    _every_epilogue_on(SMALL_16, lsa, mode, V, 64, Hq, Hkv, lens, ctx)


@pytest.mark.parametrize("D,Hq,Hkv,lens,klens", [(128, 16, 1, [742, 70, 69, 69], None), (64, 16, 16, [500, 33, 100, 64], None), (128, 40, 8, [61, 20, 8, 30, 7, 15], [148, 107, 95, 117, 94, 102])])
def test_ragged_and_short_batches_run_one_wave_per_position(lsa, D, Hq, Hkv, lens, klens):
    """Batches whose long request is counted as the only one, or as having all keys that the buffer holds beyond the rows: two waves share a tile only where a workgroup per CU is
    enough if all were as long, and where the mean request has the keys.  Which kernel ran shows in the bits: without the bound on the rows,
    or with one on the keys, the launch is one wave's without question."""
    print("case", D, Hq, Hkv, lens, flush=True)
    T, full = sum(lens), klens is None
    klens = klens or lens
    TK = sum(klens)
    q, k, v = rand_t((T, Hq, D), 61), rand_t((TK, Hkv, D), 62), rand_t((TK, Hkv, D), 63)
    qm, km = meta(lens, [0 if full else n - m for n, m in zip(klens, lens)]), meta(klens)
    o_ref, lse_ref = orc.attn_step(q, k, v, *qm, *km, 1)
    args = (*_dev(q, k, v), *_dev(*qm), *_dev(*km), 1, max(lens))
    got = lsa.prefill_attention_step(*args, total_q_len=T)
    sure = lsa.prefill_attention_step(*args) if full else lsa.prefill_attention_step(*args, total_q_len=T, max_kv_len=max(klens))
    torch.cuda.synchronize()
    assert_o_close(got[0], o_ref, "O")
    assert_lse_close(got[1], lse_ref, "LSE")
    assert torch.equal(got[0], sure[0]) and torch.equal(got[1], sure[1])


@pytest.mark.parametrize("Hq,Hkv,n,ctx", [(8, 1, 1100, 0), (4, 4, 2048, 0), (32, 8, 200, 1848), (12, 4, 77, 1300)])
def test_lone_bf16_requests_folded_in_place_are_not_copied(lsa, monkeypatch, Hq, Hkv, n, ctx):
    """The kernel of short prompts converts the V of one request of up to 2048 keys itself, through the native pass and through the checked one (which a
    bound given as a tensor takes): the same bits, and no fp16 copy of V."""
    from loongserve_amd import ops
    print("case", Hq, Hkv, n, ctx, flush=True)
    q, k, v = rand_t((n, Hq, 128), 41, torch.bfloat16), rand_t((n + ctx, Hkv, 128), 42, torch.bfloat16), rand_t((n + ctx, Hkv, 128), 43, torch.bfloat16)
    qm, km = meta([n], [ctx]), meta([n + ctx])
    o_ref, lse_ref = orc.attn_step(q, k, v, *qm, *km, 1)
    qd, kd, vd = _dev(q, k, v)
    monkeypatch.setattr(ops, "_v_as_f16", lambda *a: pytest.fail("V is copied"))
    got = []
    for bound in (n + ctx, torch.tensor(n + ctx)):
        o, m, l = torch.full_like(qd, 7.0), torch.full((n, Hq), float("-inf"), device=DEV), torch.zeros((n, Hq), device=DEV)
        lsa.context_attention_fwd(qd, kd, vd, o, *_dev(*qm), *_dev(*km), 1, n, m, l, total_q_len=n, max_kv_len=bound)
        torch.cuda.synchronize()
        assert_inplace_o_close(o.cpu(), o_ref.to(torch.bfloat16), o_ref, "o")
        assert_lse_close(orc.state_lse(m.cpu(), l.cpu()).float(), lse_ref, "state LSE")
        got.append(o)
    assert torch.equal(*got)


ROWS_256, ROWS_128, HALF = 4, 5, 6  # LSATTN_ROUTE_* of include/lsattn.h


def _in_place_on(route, lsa, V, Hq, Hkv, lens, ctx=None, full=False):
    """Prompts (behind contexts) folded in place, then the same keys once more as a step that every row sees whole (full) or as before: the route asked for as the call takes it,
    with its state, and the results against the oracle.  V: "f16" or "bf16"."""
    from loongserve_amd import _lib, ops
    dtype = torch.float16 if V == "f16" else torch.bfloat16
    ctx = ctx or [0] * len(lens)
    klens = [n + c for n, c in zip(lens, ctx)]
    T, TK = sum(lens), sum(klens)
    q, k, v = rand_t((T, Hq, 128), 31, dtype), rand_t((TK, Hkv, 128), 32, dtype), rand_t((TK, Hkv, 128), 33, dtype)
    steps = [(meta(lens, ctx), meta(klens)), (meta(lens, [2 * n for n in klens] if full else ctx), meta(klens))]
    qd, kd, vd = _dev(q, k, v)
    o, m, l = torch.full((T, Hq, 128), 7.0, dtype=dtype, device=DEV), torch.full((T, Hq), float("-inf"), device=DEV), torch.zeros((T, Hq), device=DEV)
    o_st, m_st, l_st = torch.zeros((T, Hq, 128), dtype=dtype), torch.full((T, Hq), float("-inf")), torch.zeros(T, Hq)
    parts = []
    for qm, km in steps:
        a = ops._prefill_args(qd, kd, vd, o, *_dev(*qm), *_dev(*km), 1, max(lens), None, total_q_len=T, state=(m, l))
        assert _lib.load().lsattn_prefill_route(C.byref(a)) == route
        lsa.context_attention_fwd(qd, kd, vd, o, *_dev(*qm), *_dev(*km), 1, max(lens), m, l, total_q_len=T)
        orc.context_attention_fwd(q, k, v, o_st, *qm, *km, 1, max(lens), m_st, l_st)
        parts.append(orc.attn_step(q, k, v, *qm, *km, 1))
    torch.cuda.synchronize()
    lse = torch.logaddexp(parts[0][1], parts[1][1])
    ref = sum(p[0] * (p[1] - lse).exp()[..., None] for p in parts)
    assert_inplace_o_close(o.cpu(), o_st, ref, "o")
    assert_lse_close(orc.state_lse(m.cpu(), l.cpu()).float(), lse, "state LSE")


@pytest.mark.parametrize("V,Hq,Hkv,lens,ctx,route", [
    ("f16", 8, 1, [1472], None, SMALL_16), ("f16", 24, 24, [1472], None, SMALL_16), ("f16", 8, 1, [2048], None, SMALL_16), ("bf16", 8, 1, [2048], None, SMALL_16),
    ("bf16", 4, 4, [1025], None, SMALL_16), ("f16", 32, 8, [200], [1848], SMALL_16), ("bf16", 12, 4, [77], [1300], SMALL_16), ("f16", 4, 1, [2304], None, SMALL_16),
    ("f16", 8, 8, [801] * 10, None, SMALL_32), ("f16", 8, 1, [1280] * 9, None, SMALL_32), ("f16", 18, 6, [1024] * 4, None, SMALL_32)])
def test_short_prompts_kernel_folds_in_place(lsa, V, Hq, Hkv, lens, ctx, route):
    print("case", V, Hq, Hkv, lens[:2], ctx, flush=True)
    _in_place_on(route, lsa, V, Hq, Hkv, lens, ctx)


@pytest.mark.parametrize("V", ["f16", "bf16"])
@pytest.mark.parametrize("full", [False, True])
@pytest.mark.parametrize("Hq,Hkv,lens,route", [
    (32, 8, [2500], HALF), (44, 44, [1100], HALF), (8, 1, [8300], ROWS_128), (64, 8, [800], ROWS_256),             # lone prompts past whole rounds
    (40, 8, [1600, 700, 1000, 95], HALF), (32, 8, [1400, 900, 33, 64, 1, 700, 800, 350, 555, 600], HALF), (8, 8, [900, 40, 300, 1] * 5, HALF),  # ragged: four, ten and twenty
    (16, 16, [1704, 200, 200, 200, 95], ROWS_128), (32, 8, [975, 112, 113], ROWS_256)])
def test_128_wide_kernels_shapes_fold_in_place(lsa, V, full, Hq, Hkv, lens, route):
    print("case", V, full, Hq, Hkv, lens[:4], flush=True)
    _in_place_on(route, lsa, V, Hq, Hkv, lens, full=full)
