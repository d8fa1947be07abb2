"""GPU parity of token-indexed flash decoding against the CPU oracle (through the C ABI)."""
import math

import pytest
import torch

from oracle import attn_oracle as orc
from tests.helpers import O_MAX_ABS, O_REL, assert_lse_close, assert_o_close, decode_case

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Hq,Hkv,BS", [(32, 8, 256), (4, 4, 64), (16, 8, 16), (10, 5, 128), (12, 4, 256), (8, 1, 32), (14, 2, 256),
                                       (5, 1, 64), (12, 2, 128), (3, 1, 16), (8, 1, 256), (16, 2, 64), (9, 1, 128), (32, 2, 256), (8, 2, 100), (4, 4, 7)])
def test_stage1_stage2_vs_oracle(lsa, dtype, Hq, Hkv, BS):
    _check_stage1_stage2(lsa, dtype, Hq, Hkv, BS)


def _check_stage1_stage2(lsa, dtype, Hq, Hkv, BS):
    print("case", dtype, Hq, Hkv, BS, flush=True)
    B, D = 5, 128
    lens = [700, 1, 256, 33, 1025]
    q, kv, table, b_req, b_len = decode_case(100, B, Hq, Hkv, D, lens, 3000, dtype)
    k, v = kv[:, :Hkv], kv[:, Hkv:]
    nblk = (max(lens) + BS - 1) // BS
    mid_o = torch.full((nblk, B, Hq, D), float("nan"))
    mid_l = torch.full((nblk, B, Hq), float("nan"))
    orc.decode_stage1(q, k, v, table, b_req, b_len, max(lens), mid_o, mid_l, BS)
    kvd = kv.to(DEV)
    from loongserve_amd import decoding
    # opt-in layout first: groups of blocks merged into one partial; the rows of a group's other blocks are marked empty,
    # rows past the request stay untouched, and the merge gives the same result
    assert not decoding.STAGE1_MERGES_BLOCKS  # the default is the reference's one partial per block
    decoding.STAGE1_MERGES_BLOCKS = True
    try:
        mo_d = torch.full((nblk, B, Hq, D), float("nan"), device=DEV)
        ml_d = torch.full((nblk, B, Hq), float("nan"), device=DEV)
        lsa.longserve_flash_decode_stage1(q.to(DEV), kvd[:, :Hkv], kvd[:, Hkv:], table.to(DEV), b_req.to(DEV),
                                          b_len.to(DEV), max(lens), mo_d, ml_d, BS)
    finally:
        decoding.STAGE1_MERGES_BLOCKS = False
    o_d = torch.empty(B, Hq, D, device=DEV)
    l_d = torch.empty(B, Hq, device=DEV)
    lsa.longserve_flash_decode_stage2(mo_d, ml_d, b_len.to(DEV), o_d, l_d, BS)
    torch.cuda.synchronize()
    assert torch.equal(torch.isnan(ml_d.cpu()), torch.isnan(mid_l))                 # the same rows are written
    merge = min(16, decoding._fused_block_seq(BS, B, max(lens), Hkv) // BS)
    first = (torch.arange(nblk) % merge == 0)[:, None, None]
    assert bool((torch.isinf(ml_d.cpu()) == (~first & ~torch.isnan(mid_l))).all())   # -inf exactly on a group's other rows
    o_ref, l_ref = orc.decode_full(q, k, v, table, b_req, b_len)
    assert_o_close(o_d, o_ref, "o from merged groups")
    assert_lse_close(l_d, l_ref, "lse from merged groups")
    # then the default: one partial per block, the reference's buffers
    mo_d = torch.full((nblk, B, Hq, D), float("nan"), device=DEV)
    ml_d = torch.full((nblk, B, Hq), float("nan"), device=DEV)
    lsa.longserve_flash_decode_stage1(q.to(DEV), kvd[:, :Hkv], kvd[:, Hkv:], table.to(DEV), b_req.to(DEV),
                                      b_len.to(DEV), max(lens), mo_d, ml_d, BS)
    torch.cuda.synchronize()
    # blocks past a request's length are left untouched, like the reference
    written = ~torch.isnan(mid_l)
    assert torch.equal(torch.isnan(ml_d.cpu()), ~written)
    mo_c, ml_c = mo_d.cpu(), ml_d.cpu()
    assert_o_close(torch.where(written[..., None], mo_c, torch.zeros(())), torch.where(written[..., None], mid_o, torch.zeros(())),
                   "mid_o")
    assert_lse_close(ml_c[written], mid_l[written], "mid_lse")
    for odt in (torch.float32, dtype):
        o_d = torch.empty(B, Hq, D, dtype=odt, device=DEV)
        l_d = torch.empty(B, Hq, device=DEV)
        lsa.longserve_flash_decode_stage2(mo_d, ml_d, b_len.to(DEV), o_d, l_d, BS)
        torch.cuda.synchronize()
        o_ref, l_ref = orc.decode_full(q, k, v, table, b_req, b_len)
        if odt == torch.bfloat16:
            assert_o_close(o_d, o_ref, "o bf16 out", max_abs=4e-3, rel=4e-3)  # 8-bit mantissa output
        else:
            assert_o_close(o_d, o_ref, "o")
        assert_lse_close(l_d, l_ref, "lse")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("merge", [2, 8, 16])
@pytest.mark.parametrize("Hq,Hkv,BS,lens", [
    (32, 8, 16, [700, 1, 256, 33, 1025]),      # group 4, many short blocks
    (8, 1, 128, [5000]),                       # group 8 (two rounds of four heads), one request: the waves split a block
    (16, 1, 256, [3000, 9000]),                # group 16 (two tasks per KV head), few workgroups: split path
    (16, 4, 32, [100, 2049, 17, 640, 1, 999]),  # group 4, ragged
    (4, 4, 128, [4097, 130]),                  # one query head per KV head
])
def test_stage1_forced_merge_blocks(lsa, dtype, merge, Hq, Hkv, BS, lens):
    _check_merge_blocks(lsa, dtype, merge, Hq, Hkv, BS, lens)


def _check_merge_blocks(lsa, dtype, merge, Hq, Hkv, BS, lens):
    """merge_blocks = m of flash_decoding_stage1: the partial of blocks [m j, m j + m) of a request in row m j, the other
    rows the request reaches marked empty, rows past it untouched; checked row by row against the oracle's stage 1 at
    block size m * BS, and through stage 2 at the caller's block size."""
    print("case", dtype, merge, Hq, Hkv, BS, lens, flush=True)
    B, D = len(lens), 128
    q, kv, table, b_req, b_len = decode_case(500 + merge, B, Hq, Hkv, D, lens, sum(lens) + 300, dtype)
    k, v = kv[:, :Hkv], kv[:, Hkv:]
    nblk = (max(lens) + BS - 1) // BS
    ngrp = (nblk + merge - 1) // merge
    ref_o = torch.full((ngrp, B, Hq, D), float("nan"))
    ref_l = torch.full((ngrp, B, Hq), float("nan"))
    orc.decode_stage1(q, k, v, table, b_req, b_len, max(lens), ref_o, ref_l, BS * merge)
    kvd = kv.to(DEV)
    mo_d = torch.full((nblk, B, Hq, D), float("nan"), device=DEV)
    ml_d = torch.full((nblk, B, Hq), float("nan"), device=DEV)
    lsa.longserve_cuda_kernels.flash_decoding_stage1(mo_d, ml_d, q.to(DEV), kvd[:, :Hkv], kvd[:, Hkv:], table.to(DEV), b_req.to(DEV),
                                                     b_len.to(DEV), max(lens), BS, merge)
    torch.cuda.synchronize()
    mo_c, ml_c = mo_d.cpu(), ml_d.cpu()
    for b in range(B):
        reach = (lens[b] + BS - 1) // BS
        for i in range(nblk):
            if i >= reach:
                assert torch.isnan(ml_c[i, b]).all() and torch.isnan(mo_c[i, b]).all(), (b, i)   # untouched
            elif i % merge:
                assert (ml_c[i, b] == float("-inf")).all() and torch.isnan(mo_c[i, b]).all(), (b, i)  # empty, mid_o left alone
            else:
                assert_o_close(mo_c[i, b], ref_o[i // merge, b], "mid_o row %d request %d" % (i, b))
                assert_lse_close(ml_c[i, b], ref_l[i // merge, b], "mid_lse row %d request %d" % (i, b))
    o_d = torch.empty(B, Hq, D, device=DEV)
    l_d = torch.empty(B, Hq, device=DEV)
    lsa.longserve_flash_decode_stage2(mo_d, ml_d, b_len.to(DEV), o_d, l_d, BS)
    torch.cuda.synchronize()
    o_ref, l_ref = orc.decode_full(q, k, v, table, b_req, b_len)
    assert_o_close(o_d, o_ref, "o")
    assert_lse_close(l_d, l_ref, "lse")


@pytest.fixture(params=["mfma", "split", "mfma listed"], ids=["plain", "split", "listed"])
def matrix_pipe(tuning, request):
    """Stage 1 through the matrix-pipe kernel wherever its conditions hold, whatever the launch's size: its plain shape
    (a wave per 256 tokens; blocks a multiple of 32 tokens; by itself the library takes it for large launches), the
    shape whose four waves split a block (blocks a multiple of 128 tokens; small launches of groups of four and more),
    and the plain shape over a list of the units that exist (by itself: launches of very many workgroups)."""
    tuning(decode_stage1=request.param.split()[0], decode_listed="on" if "listed" in request.param else "off")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Hq,Hkv,BS", [(32, 8, 256), (4, 4, 64), (10, 5, 128), (8, 1, 32), (5, 1, 64), (9, 1, 128), (16, 2, 64), (32, 2, 256),
                                       (17, 1, 96), (66, 2, 32), (7, 7, 160)])
def test_matrix_pipe_stage1_stage2_vs_oracle(lsa, matrix_pipe, dtype, Hq, Hkv, BS):
    """Groups of 1 to 33 query heads (padded to 16-row operands, 17 and 33: a second / third task with one live row),
    blocks of one to eight 32-token batches, requests of 1 token, of a partial batch and of a partial block."""
    _check_stage1_stage2(lsa, dtype, Hq, Hkv, BS)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("merge", [2, 16])
@pytest.mark.parametrize("Hq,Hkv,BS,lens", [
    (8, 1, 128, [5000]),
    (16, 1, 256, [3000, 9000]),
    (16, 4, 32, [100, 2049, 17, 640, 1, 999]),
    (40, 8, 64, [4097, 130]),
])
def test_matrix_pipe_stage1_forced_merge_blocks(lsa, matrix_pipe, dtype, merge, Hq, Hkv, BS, lens):
    _check_merge_blocks(lsa, dtype, merge, Hq, Hkv, BS, lens)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_large_group_launch_that_takes_the_matrix_pipe_by_itself(lsa, dtype):
    """64 query heads over 8 KV heads, 2 requests of about 17000 tokens: 2 x 8 x 67 waves of the matrix-pipe kernel, the
    library's own choice (nothing forced), through the fused call and through the two stages."""
    lsa.set_tuning()
    B, Hq, Hkv, D, BS = 2, 64, 8, 128, 256
    lens = [17000, 16411]
    q, kv, table, b_req, b_len = decode_case(77, B, Hq, Hkv, D, lens, sum(lens) + 1000, dtype)
    k, v = kv[:, :Hkv], kv[:, Hkv:]
    o_ref, l_ref = orc.decode_full(q, k, v, table, b_req, b_len)
    kvd = kv.to(DEV)
    nblk = (max(lens) + BS - 1) // BS
    mo_d = torch.full((nblk, B, Hq, D), float("nan"), device=DEV)
    ml_d = torch.full((nblk, B, Hq), float("nan"), device=DEV)
    o_d = torch.empty(B, Hq, D, device=DEV)
    l_d = torch.empty(B, Hq, device=DEV)
    lsa.longserve_token_decode_attention_flash_decoding(q.to(DEV), table.to(DEV), b_req.to(DEV), b_len.to(DEV), mo_d, ml_d, B, max(lens),
                                                        Hq, D, kvd[:, :Hkv], kvd[:, Hkv:], BS, o_d, l_d)
    torch.cuda.synchronize()
    assert_o_close(o_d, o_ref, "o, fused call")
    assert_lse_close(l_d, l_ref, "lse, fused call")
    mo_d.fill_(float("nan"))
    ml_d.fill_(float("nan"))
    lsa.longserve_flash_decode_stage1(q.to(DEV), kvd[:, :Hkv], kvd[:, Hkv:], table.to(DEV), b_req.to(DEV), b_len.to(DEV), max(lens),
                                      mo_d, ml_d, BS)
    lsa.longserve_flash_decode_stage2(mo_d, ml_d, b_len.to(DEV), o_d, l_d, BS)
    torch.cuda.synchronize()
    reach = torch.tensor([(n + BS - 1) // BS for n in lens])
    assert torch.equal(torch.isnan(ml_d.cpu()), (torch.arange(nblk)[:, None] >= reach[None, :])[:, :, None].expand(nblk, B, Hq))
    assert_o_close(o_d, o_ref, "o, two stages")
    assert_lse_close(l_d, l_ref, "lse, two stages")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_skewed_batch_that_walks_the_unit_list_by_itself(lsa, dtype):
    """One request of 40000 tokens among 127 of 1 to 300 (and two of none), 64 tokens per partial: the plain grid would
    be 157 x 2 x 130 = 40820 workgroups, nearly all of them without work, so the library walks the list of the units
    that exist (its own choice: nothing forced).  Two stages, per-block partials; rows no request reaches stay
    untouched."""
    lsa.set_tuning()
    import random
    rng = random.Random(5)
    B, Hq, Hkv, D, BS = 130, 32, 8, 128, 64
    lens = [rng.randint(1, 300) for _ in range(B)]
    lens[37] = 40000
    lens[0] = lens[129] = lens[64] = 0
    lens[1] = 64
    q, kv, table, b_req, b_len = decode_case(78, B, Hq, Hkv, D, lens, sum(lens) + 1000, dtype)
    k, v = kv[:, :Hkv], kv[:, Hkv:]
    live = [b for b in range(B) if lens[b] > 0]
    o_ref, l_ref = orc.decode_full(q[live], k, v, table, b_req[live], b_len[live])
    kvd = kv.to(DEV)
    nblk = (max(lens) + BS - 1) // BS
    mo_d = torch.full((nblk, B, Hq, D), float("nan"), device=DEV)
    ml_d = torch.full((nblk, B, Hq), float("nan"), device=DEV)
    o_d = torch.empty(B, Hq, D, device=DEV)
    l_d = torch.empty(B, Hq, device=DEV)
    lsa.longserve_flash_decode_stage1(q.to(DEV), kvd[:, :Hkv], kvd[:, Hkv:], table.to(DEV), b_req.to(DEV), b_len.to(DEV), max(lens),
                                      mo_d, ml_d, BS)
    lsa.longserve_flash_decode_stage2(mo_d, ml_d, b_len.to(DEV), o_d, l_d, BS)
    torch.cuda.synchronize()
    reach = torch.tensor([(n + BS - 1) // BS for n in lens])
    assert torch.equal(torch.isnan(ml_d.cpu()), (torch.arange(nblk)[:, None] >= reach[None, :])[:, :, None].expand(nblk, B, Hq))
    assert_o_close(o_d[live], o_ref, "o, two stages")
    assert_lse_close(l_d[live], l_ref, "lse, two stages")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_fused_call_gives_the_same_bits_with_either_layout_of_its_partials(lsa, monkeypatch, dtype):
    """The fused call keeps the partials of a request side by side in mid_o; with the reference's layout (a block of all
    requests after the other, what the two stage functions use) it must return the same bits."""
    B, Hq, Hkv, D, BS = 5, 16, 4, 128, 64
    lens = [700, 1, 64, 2049, 333]
    q, kv, table, b_req, b_len = decode_case(91, B, Hq, Hkv, D, lens, sum(lens) + 100, dtype)
    o_ref, l_ref = orc.decode_full(q, kv[:, :Hkv], kv[:, Hkv:], table, b_req, b_len)
    kvd = kv.to(DEV)
    nblk = (max(lens) + BS - 1) // BS
    res = []
    for by_request in (True, False):
        monkeypatch.setattr(lsa.longserve_cuda_kernels, "FUSED_PARTIALS_BY_REQUEST", by_request)
        mo_d = torch.full((nblk, B, Hq, D), float("nan"), device=DEV)
        ml_d = torch.full((nblk, B, Hq), float("nan"), device=DEV)
        o_d = torch.empty(B, Hq, D, device=DEV)
        l_d = torch.empty(B, Hq, device=DEV)
        lsa.longserve_cuda_kernels.flash_decoding(mo_d, ml_d, q.to(DEV), kvd[:, :Hkv], kvd[:, Hkv:], table.to(DEV), b_req.to(DEV),
                                                  b_len.to(DEV), max(lens), o_d, l_d, BS)
        torch.cuda.synchronize()
        assert_o_close(o_d, o_ref, "o, partials by request %s" % by_request)
        assert_lse_close(l_d, l_ref, "lse, partials by request %s" % by_request)
        res.append((o_d.cpu(), l_d.cpu(), ml_d.cpu()))
    assert torch.equal(res[0][0], res[1][0]) and torch.equal(res[0][1], res[1][1])
    # the same partials, in the other order: request b's block i is row (b, i) of the one and row (i, b) of the other
    by_req = res[0][2].reshape(B, nblk, Hq)
    for b, n in enumerate(lens):
        for i in range((n + BS - 1) // BS):
            assert torch.equal(by_req[b, i], res[1][2][i, b]), (b, i)


@pytest.mark.parametrize("B", [1024, 1025])
def test_unit_list_at_its_largest_batch_and_past_it(lsa, tuning, B):
    """The list of units is numbered in LDS for up to 1024 requests; a larger batch takes the plain grid whatever the
    tuning block asks for.  Requests of 0 to 120 tokens and one of 9000, 64 tokens per partial."""
    import random
    tuning(decode_stage1="mfma", decode_listed="on")
    rng = random.Random(B)
    Hq, Hkv, D, BS = 8, 2, 128, 64
    lens = [rng.randint(0, 120) for _ in range(B)]
    lens[B // 3] = 9000
    q, kv, table, b_req, b_len = decode_case(500 + B, B, Hq, Hkv, D, lens, sum(lens) + 300)
    o_ref, l_ref = orc.decode_full(q, kv[:, :Hkv], kv[:, Hkv:], table, b_req, b_len)
    kvd = kv.to(DEV)
    nblk = (max(lens) + BS - 1) // BS
    mo_d = torch.full((nblk, B, Hq, D), float("nan"), device=DEV)
    ml_d = torch.full((nblk, B, Hq), float("nan"), device=DEV)
    lsa.longserve_flash_decode_stage1(q.to(DEV), kvd[:, :Hkv], kvd[:, Hkv:], table.to(DEV), b_req.to(DEV), b_len.to(DEV), max(lens),
                                      mo_d, ml_d, BS)
    o_d = torch.empty(B, Hq, D, device=DEV)
    l_d = torch.empty(B, Hq, device=DEV)
    lsa.longserve_flash_decode_stage2(mo_d, ml_d, b_len.to(DEV), o_d, l_d, BS)
    torch.cuda.synchronize()
    live = [b for b in range(B) if lens[b] > 0]
    reach = torch.tensor([(n + BS - 1) // BS for n in lens])
    assert torch.equal(torch.isnan(ml_d.cpu()), (torch.arange(nblk)[:, None] >= reach[None, :])[:, :, None].expand(nblk, B, Hq))
    assert_o_close(o_d[live], o_ref[live], "o")
    assert_lse_close(l_d[live], l_ref[live], "lse")


def test_gather_indices_bit_exact(lsa):
    # q = 0 and V[slot] = ordinal code of the slot: the set of gathered slots is read back from O*len
    B, H, D = 3, 2, 128
    lens = [37, 300, 1000]
    q, kv, table, b_req, b_len = decode_case(200, B, H, H, D, lens, 1500)
    q.zero_()
    kv[:, H:, :] = (torch.arange(1500, dtype=torch.float32) % 2048)[:, None, None].to(torch.float16)
    kv[:, H:, 1] = 1.0
    kvd = kv.to(DEV)
    BS = 256
    nblk = (max(lens) + BS - 1) // BS
    mo = torch.zeros(nblk, B, H, D, device=DEV)
    ml = torch.zeros(nblk, B, H, device=DEV)
    o, lse = lsa.longserve_token_decode_attention_flash_decoding(q.to(DEV), table.to(DEV), b_req.to(DEV), b_len.to(DEV),
                                                                 mo, ml, B, max(lens), H, D, kvd[:, :H], kvd[:, H:], BS)
    torch.cuda.synchronize()
    assert o.dtype == torch.float32
    for b in range(B):
        slots = table[int(b_req[b]), :lens[b]].long()
        want = float(kv[slots, H, 0].float().sum())
        got = float(o[b, 0, 0]) * lens[b]
        assert abs(got - want) <= 1e-4 * max(want, 1.0) + 0.5, (got, want)
        assert abs(float(o[b, 1, 1]) - 1.0) < 1e-6
        assert abs(float(lse[b, 0]) - math.log(lens[b])) < 1e-5


def test_multi_instance_decode_with_empty_peer(lsa):
    # each request's KV split over 3 instances; one peer holds nothing for one request
    from loongserve_amd.simulate import DecodeInstance, multi_instance_decode
    B, Hq, Hkv, D = 4, 8, 2, 128
    lens = [900, 64, 333, 2000]
    q, kv, table, b_req, b_len = decode_case(300, B, Hq, Hkv, D, lens, 4000)
    o_ref, l_ref = orc.decode_full(q, kv[:, :Hkv], kv[:, Hkv:], table, b_req, b_len)
    cuts = [[300, 600], [0, 64], [111, 111], [700, 1300]]  # ranges: master [0,c0), peer1 [c0,c1), peer2 [c1,len)
    kvd = kv.to(DEV)
    insts = []
    for r in range(3):
        t = torch.full_like(table, orc.INT32_PAD)
        ln = []
        for b in range(B):
            lo = [0, cuts[b][0], cuts[b][1]][r]
            hi = [cuts[b][0], cuts[b][1], lens[b]][r]
            t[int(b_req[b]), :hi - lo] = table[int(b_req[b]), lo:hi]
            ln.append(hi - lo)
        insts.append(DecodeInstance(kvd, t.to(DEV), b_req.to(DEV), torch.tensor(ln, dtype=torch.int32, device=DEV), max(ln)))
    o, lse = multi_instance_decode(q.to(DEV), insts, Hkv)
    torch.cuda.synchronize()
    assert o.dtype == torch.float16
    assert_o_close(o, o_ref, "multi-instance o")
    assert_lse_close(lse, l_ref, "multi-instance lse")


def test_stage2_empty_request_defined(lsa):
    B, H, D = 2, 4, 128
    mo = torch.randn(3, B, H, D, device=DEV)
    ml = torch.randn(3, B, H, device=DEV)
    o = torch.full((B, H, D), 7.0, device=DEV)
    l = torch.full((B, H), 7.0, device=DEV)
    lsa.longserve_flash_decode_stage2(mo, ml, torch.tensor([0, 3], dtype=torch.int32, device=DEV), o, l, 1)
    torch.cuda.synchronize()
    assert torch.all(o[0] == 0) and torch.all(torch.isinf(l[0]) & (l[0] < 0))
    o_ref, l_ref = orc.lse_merge([(mo[i, 1].cpu(), ml[i, 1].cpu()) for i in range(3)])
    assert_o_close(o[1], o_ref, "o", max_abs=1e-5, rel=1e-5)
    assert_lse_close(l[1], l_ref, "lse", rel=1e-5)


@pytest.mark.parametrize("lead", [0, 1, 3, 70])
@pytest.mark.parametrize("own", [1, 5, 66])
def test_stage2_with_rows_of_peers_in_front(lsa, lead, own):
    """The peers' rows and a request's own blocks, whose number follows from its length: as the merge of so many rows of one token each."""
    print("case", lead, own, flush=True)
    B, H, D, BS = 5, 3, 128, 16
    g = torch.Generator().manual_seed(lead * 100 + own)
    mo, ml = torch.randn(lead + own, B, H, D, generator=g).to(DEV), torch.randn(lead + own, B, H, generator=g).to(DEV)
    lens = torch.tensor([own * BS, 0, 1, (own * BS) // 2 + 1, 3 * own * BS], dtype=torch.int32)  # (the last one: no more rows than there are)
    rows = torch.tensor([own, 0, 1, -(-((own * BS) // 2 + 1) // BS), own], dtype=torch.int32) + lead
    got = []
    for args in ((lens, BS, lead), (rows, 1)):
        o, l = torch.full((B, H, D), 9.0, device=DEV), torch.full((B, H), 9.0, device=DEV)
        lsa.longserve_flash_decode_stage2(mo, ml, args[0].to(DEV), o, l, *args[1:])
        got.append((o, l))
    torch.cuda.synchronize()
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    with pytest.raises(ValueError):
        lsa.longserve_flash_decode_stage2(mo, ml, lens.to(DEV), o, l, BS, -1)


@pytest.mark.parametrize("nblk", [1, 7, 31, 64, 65, 300, 1029])
def test_stage2_alone_over_few_and_many_partials(lsa, nblk):
    """The merge on its own, on random partials: every count of blocks around the points where the kernel changes its
    walk (rows in flight per slice, the wide launch for many partials of few rows), empty partials in between, requests
    that use fewer blocks than the buffer has, fp32 and fp16 outputs."""
    print("case nblk", nblk, flush=True)
    B, H, D, BS = 3, 5, 128, 16
    g = torch.Generator().manual_seed(nblk)
    mo = torch.randn(nblk, B, H, D, generator=g)
    ml = torch.randn(nblk, B, H, generator=g) * 6
    ml[torch.rand(nblk, B, H, generator=g) < 0.15] = float("-inf")
    lens = torch.tensor([nblk * BS, max(1, (nblk * BS) // 3 + 1), 0], dtype=torch.int32)
    o_ref = torch.empty(B, H, D)
    l_ref = torch.empty(B, H)
    orc.decode_stage2(mo, ml, lens, o_ref, l_ref, BS)
    for odt in (torch.float32, torch.float16):
        o = torch.full((B, H, D), 9.0, dtype=odt, device=DEV)
        l = torch.full((B, H), 9.0, device=DEV)
        lsa.longserve_flash_decode_stage2(mo.to(DEV), ml.to(DEV), lens.to(DEV), o, l, BS)
        torch.cuda.synchronize()
        # a (b, h) whose partials are all empty merges to (0, -inf), like a request without tokens
        dead = torch.isinf(l_ref) & (l_ref < 0)
        assert torch.equal(torch.isinf(l.cpu()) & (l.cpu() < 0), dead)
        assert torch.all(o.cpu()[dead] == 0)
        if odt == torch.float32:
            assert_o_close(o, torch.where(dead[..., None], torch.zeros(()), o_ref), "o", max_abs=2e-5, rel=1e-5)
        else:
            assert_o_close(o, torch.where(dead[..., None], torch.zeros(()), o_ref), "o fp16", max_abs=4e-3, rel=1e-3)
        assert_lse_close(l, l_ref, "lse", rel=1e-5)


@pytest.mark.parametrize("B,H,nblk", [(70, 32, 1030), (300, 8, 520), (9, 5, 1024)])
def test_stage2_of_one_long_request_among_many_short_ones(lsa, B, H, nblk):
    """The merge of a batch in which one request has a thousand partials and the others a few: more (request, head) pairs
    than the narrow launch's bound for the wide one, with enough partials for the wide launch all the same (70 x 32), too
    many pairs for it (300 x 8), and a small batch; the long request in the middle of the batch, so that the heads of a
    request and the requests of a head are both told apart in the grid."""
    print("case", B, H, nblk, flush=True)
    D, BS = 128, 16
    g = torch.Generator().manual_seed(B * 1000 + nblk)
    mo = torch.randn(nblk, B, H, D, generator=g)
    ml = torch.randn(nblk, B, H, generator=g) * 5
    ml[torch.rand(nblk, B, H, generator=g) < 0.1] = float("-inf")
    lens = torch.randint(1, 4 * BS, (B,), generator=g).to(torch.int32)
    lens[B // 2] = nblk * BS - 3
    lens[0] = 0
    o_ref = torch.empty(B, H, D)
    l_ref = torch.empty(B, H)
    orc.decode_stage2(mo, ml, lens, o_ref, l_ref, BS)
    o = torch.full((B, H, D), 9.0, device=DEV)
    l = torch.full((B, H), 9.0, device=DEV)
    lsa.longserve_flash_decode_stage2(mo.to(DEV), ml.to(DEV), lens.to(DEV), o, l, BS)
    torch.cuda.synchronize()
    dead = torch.isinf(l_ref) & (l_ref < 0)
    assert torch.equal(torch.isinf(l.cpu()) & (l.cpu() < 0), dead)
    assert_o_close(o, torch.where(dead[..., None], torch.zeros(()), o_ref), "o", max_abs=2e-5, rel=1e-5)
    assert_lse_close(l, l_ref, "lse", rel=1e-5)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_peaked_softmax_keeps_the_bars(lsa, dtype):
    """Scores of magnitude up to ~64: a few tokens carry each request."""
    B, Hq, Hkv, D, BS = 3, 4, 2, 128, 256
    lens = [3000, 700, 64]
    q, kv, table, b_req, b_len = decode_case(5, B, Hq, Hkv, D, lens, 5000, dtype)
    g = torch.Generator().manual_seed(9)
    q = (torch.randn(q.shape, generator=g) * 4).to(dtype)
    kv[:, :Hkv] = (torch.randn((5000, Hkv, D), generator=g) * 4).to(dtype)
    o_ref, l_ref = orc.decode_full(q, kv[:, :Hkv], kv[:, Hkv:], table, b_req, b_len)
    kvd = kv.to(DEV)
    nblk = (max(lens) + BS - 1) // BS
    mo = torch.empty(nblk, B, Hq, D, device=DEV)
    ml = torch.empty(nblk, B, Hq, device=DEV)
    o, l = lsa.longserve_token_decode_attention_flash_decoding(q.to(DEV), table.to(DEV), b_req.to(DEV), b_len.to(DEV), mo, ml, B,
                                                               max(lens), Hq, D, kvd[:, :Hkv], kvd[:, Hkv:], BS)
    torch.cuda.synchronize()
    assert_o_close(o, o_ref, "o")
    assert_lse_close(l, l_ref, "lse")


def test_one_request_of_a_million_tokens(lsa):
    """The longest context the serving configs name (1M tokens) in one request: the fused call's coarsest split, the wide
    merge, 32-bit positions near 2^20 and slot numbers above 2^20.  Checked through closed forms rather than a CPU pass
    over 1 GB of rows: q = 0 gives O = mean of the request's V rows and LSE = ln(n); a query equal to 40 x one key's
    direction puts almost all weight on that token."""
    n, Hq, Hkv, D, BS = 1_048_576, 4, 2, 128, 256
    pool = n + 4096
    g = torch.Generator(device=DEV).manual_seed(11)
    kv = (torch.randn((pool, 2 * Hkv, D), generator=g, device=DEV) * 0.5).half()
    perm = torch.randperm(pool, generator=g, device=DEV)[:n].to(torch.int32)
    table = torch.full((2, n + 8), 2147483647, dtype=torch.int32, device=DEV)
    table[1, :n] = perm
    b_req = torch.tensor([1], dtype=torch.int32, device=DEV)
    b_len = torch.tensor([n], dtype=torch.int32, device=DEV)
    nblk = (n + BS - 1) // BS
    mo = torch.empty(nblk, 1, Hq, D, device=DEV)
    ml = torch.empty(nblk, 1, Hq, device=DEV)
    q = torch.zeros(1, Hq, D, dtype=torch.float16, device=DEV)
    o, lse = lsa.longserve_token_decode_attention_flash_decoding(q, table, b_req, b_len, mo, ml, 1, n, Hq, D, kv[:, :Hkv], kv[:, Hkv:], BS)
    torch.cuda.synchronize()
    v_mean = kv[perm.long(), Hkv:].double().mean(0)                        # [Hkv, D]
    want = v_mean.repeat_interleave(Hq // Hkv, 0)[None].float()
    assert (o - want).abs().max().item() <= 2e-5
    assert (lse - math.log(n)).abs().max().item() <= 1e-4 * math.log(n)
    # a peaked query: token t of the request (any position, here near the end) dominates
    t = n - 12345
    slot = int(perm[t])
    kdir = kv[slot, :Hkv].float()                                          # [Hkv, D]
    q2 = (kdir * (40.0 / kdir.norm(dim=-1, keepdim=True))).repeat_interleave(Hq // Hkv, 0)[None].half()
    o2, lse2 = lsa.longserve_token_decode_attention_flash_decoding(q2, table, b_req, b_len, mo, ml, 1, n, Hq, D, kv[:, :Hkv], kv[:, Hkv:], BS)
    torch.cuda.synchronize()
    s = torch.einsum("hd,nhd->hn", q2[0].float().view(Hkv, Hq // Hkv, D).reshape(Hq, D)[::Hq // Hkv], kv[perm.long(), :Hkv].float()) / math.sqrt(D)
    lse_ref = torch.logsumexp(s.double(), dim=-1).float().repeat_interleave(Hq // Hkv)
    o_ref = torch.einsum("hn,nhd->hd", torch.softmax(s.double(), dim=-1), kv[perm.long(), Hkv:].double()).float().repeat_interleave(Hq // Hkv, 0)
    assert_lse_close(lse2[0], lse_ref.cpu(), "peaked lse")
    assert_o_close(o2[0], o_ref.cpu(), "peaked o")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Hq,Hkv,BS,lens", [
    (32, 8, 256, [5000, 1, 256, 257, 0, 9000, 300]),          # two task groups of four KV heads
    (8, 1, 256, [3000, 700, 12000, 256]),                     # one KV head: the four waves of a workgroup hold four shares
    (16, 2, 512, [100, 5000, 2049, 17, 1024, 1, 999]),        # two KV heads: two waves on tasks, two shares per workgroup
    (40, 5, 256, [4097, 130, 0, 0, 6000]),                    # five KV heads: the second task group half empty
    (17, 1, 1024, [40000, 3, 2048]),                          # a second task with one live row; a split of 1024 dealt in blocks of 256
])
def test_fused_call_in_equal_shares(lsa, tuning, dtype, Hq, Hkv, BS, lens):
    """The fused call with stage 1 dealt in equal shares of blocks (forced: these launches are far smaller than the ones
    the library deals that way by itself): shares that end inside a request, requests inside a share, requests without
    tokens, more workers than blocks; the partials' buffers start as NaN (every row the merge reads must have been
    written, as a partial or as an empty row) and are as tall as the caller's BLOCK_SEQ of 256 makes them."""
    tuning(decode_listed="shares")
    B, D = len(lens), 128
    q, kv, table, b_req, b_len = decode_case(500 + Hq + len(lens), B, Hq, Hkv, D, lens, sum(lens) + 500, dtype)
    o_ref, l_ref = orc.decode_full(q, kv[:, :Hkv], kv[:, Hkv:], table, b_req, b_len)
    kvd = kv.to(DEV)
    nblk = (max(lens) + 255) // 256
    mo_d = torch.full((nblk, B, Hq, D), float("nan"), device=DEV)
    ml_d = torch.full((nblk, B, Hq), float("nan"), device=DEV)
    o_d = torch.full((B, Hq, D), float("nan"), device=DEV)
    l_d = torch.full((B, Hq), float("nan"), device=DEV)
    lsa.longserve_cuda_kernels.flash_decoding(mo_d, ml_d, q.to(DEV), kvd[:, :Hkv], kvd[:, Hkv:], table.to(DEV), b_req.to(DEV), b_len.to(DEV),
                                              max(lens), o_d, l_d, BS)
    torch.cuda.synchronize()
    assert_o_close(o_d, o_ref, "o")
    assert_lse_close(l_d, l_ref, "lse")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_large_batch_that_is_dealt_in_equal_shares_by_itself(lsa, dtype):
    """48 requests of 1 to 9000 tokens, 32 query heads on 8 KV heads: 48 x 36 blocks of 256 tokens at most, enough for the
    library to deal them in equal shares by itself (nothing forced) in the fused call; the two stages on their own keep
    one partial per block."""
    lsa.set_tuning()
    import random
    rng = random.Random(17)
    B, Hq, Hkv, D, BS = 48, 32, 8, 128, 256
    lens = [rng.randint(1, 9000) for _ in range(B)]
    lens[5] = 9000
    lens[6] = 0
    q, kv, table, b_req, b_len = decode_case(79, B, Hq, Hkv, D, lens, sum(lens) + 1000, dtype)
    o_ref, l_ref = orc.decode_full(q, kv[:, :Hkv], kv[:, Hkv:], table, b_req, b_len)
    kvd = kv.to(DEV)
    nblk = (max(lens) + BS - 1) // BS
    mo_d = torch.full((nblk, B, Hq, D), float("nan"), device=DEV)
    ml_d = torch.full((nblk, B, Hq), float("nan"), device=DEV)
    o_d = torch.empty(B, Hq, D, device=DEV)
    l_d = torch.empty(B, Hq, device=DEV)
    lsa.longserve_token_decode_attention_flash_decoding(q.to(DEV), table.to(DEV), b_req.to(DEV), b_len.to(DEV), mo_d, ml_d, B, max(lens),
                                                        Hq, D, kvd[:, :Hkv], kvd[:, Hkv:], BS, o_d, l_d)
    torch.cuda.synchronize()
    assert_o_close(o_d, o_ref, "o, fused call")
    assert_lse_close(l_d, l_ref, "lse, fused call")
    # (in equal shares a request has far fewer partials than blocks: most rows of the buffer are never written)
    ml = ml_d.cpu()
    assert int(torch.isnan(ml).sum()) > int(torch.isfinite(ml).sum()) > 0
    # the entry point that brings its own partials takes the same route (its array holds a row per 256 tokens here)
    o_s = torch.full((B, Hq, D), float("nan"), device=DEV)
    l_s = torch.full((B, Hq), float("nan"), device=DEV)
    lsa.longserve_cuda_kernels.flash_decoding_static(q.to(DEV), kvd[:, :Hkv], kvd[:, Hkv:], table.to(DEV), b_req.to(DEV), b_len.to(DEV),
                                                     max(lens), o_s, l_s, 1024)
    torch.cuda.synchronize()
    assert torch.equal(o_s, o_d) and torch.equal(l_s, l_d)
    # recorded in a HIP graph and replayed on new queries: every replay against the eager call
    qd = q.to(DEV).clone()
    td, rd, ld = table.to(DEV), b_req.to(DEV), b_len.to(DEV)
    o_g = torch.empty(B, Hq, D, device=DEV)
    l_g = torch.empty(B, Hq, device=DEV)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        lsa.longserve_token_decode_attention_flash_decoding(qd, td, rd, ld, mo_d, ml_d, B, max(lens), Hq, D, kvd[:, :Hkv], kvd[:, Hkv:], BS, o_g, l_g)
    for rep in range(3):
        qd.copy_((torch.randn(q.shape, generator=torch.Generator().manual_seed(900 + rep)) * 0.5).to(dtype))
        o_g.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        o_e = torch.empty(B, Hq, D, device=DEV)
        l_e = torch.empty(B, Hq, device=DEV)
        lsa.longserve_token_decode_attention_flash_decoding(qd, td, rd, ld, mo_d, ml_d, B, max(lens), Hq, D, kvd[:, :Hkv], kvd[:, Hkv:], BS, o_e, l_e)
        torch.cuda.synchronize()
        assert torch.equal(o_g, o_e) and torch.equal(l_g, l_e), "replay %d" % rep


@pytest.mark.parametrize("seed", [5, 19, 77])
def test_random_fused_calls_in_equal_shares(lsa, tuning, seed):
    """Seeded random sweep of the fused call with stage 1 forced into equal shares, and of the entry point that brings
    its own partials on the same inputs (bit for bit the same where the caller's buffers are tall enough for blocks of
    256 tokens, which is what that entry point always deals): 1 to 40 requests of 0 to 9000 tokens (several empty,
    of one token, of exactly a block), groups of 1 to 20 query heads on 1 to 8 KV heads, both dtypes, the caller's
    BLOCK_SEQ 256 to 2048, buffers as tall as that makes them."""
    import random
    rng = random.Random(seed)
    tuning(decode_listed="shares")
    for case in range(8):
        dtype = rng.choice([torch.float16, torch.bfloat16])
        Hkv = rng.choice([1, 2, 3, 5, 8])
        Hq = Hkv * rng.choice([1, 2, 4, 5, 8, 16, 17, 20])
        BS = rng.choice([256, 512, 1024, 2048])
        B = rng.choice([1, 2, 3, 9, 17, 40])
        lens = [rng.choice([0, 1, 2, 255, 256, 257, 511, 512, 1000, 2049, 4096, 9000, rng.randint(1, 9000)]) for _ in range(B)]
        if max(lens) == 0:
            lens[0] = 300
        print("case", seed, case, dtype, Hq, Hkv, BS, lens, flush=True)
        D = 128
        q, kv, table, b_req, b_len = decode_case(7000 + 100 * seed + case, B, Hq, Hkv, D, lens, sum(lens) + 300, dtype)
        o_ref, l_ref = orc.decode_full(q, kv[:, :Hkv], kv[:, Hkv:], table, b_req, b_len)
        kvd, qd, td, rd, ld = kv.to(DEV), q.to(DEV), table.to(DEV), b_req.to(DEV), b_len.to(DEV)
        nblk = (max(lens) + BS - 1) // BS
        mo_d = torch.full((nblk, B, Hq, D), float("nan"), device=DEV)
        ml_d = torch.full((nblk, B, Hq), float("nan"), device=DEV)
        o_d = torch.full((B, Hq, D), float("nan"), device=DEV)
        l_d = torch.full((B, Hq), float("nan"), device=DEV)
        lsa.longserve_cuda_kernels.flash_decoding(mo_d, ml_d, qd, kvd[:, :Hkv], kvd[:, Hkv:], td, rd, ld, max(lens), o_d, l_d, BS)
        torch.cuda.synchronize()
        what = "seed %d case %d" % (seed, case)
        live = torch.tensor(lens) > 0
        assert_o_close(o_d[live.to(DEV)], o_ref[live], "o, " + what)
        assert_lse_close(l_d, l_ref, "lse, " + what)
        o_s = torch.full((B, Hq, D), float("nan"), device=DEV)
        l_s = torch.full((B, Hq), float("nan"), device=DEV)
        lsa.longserve_cuda_kernels.flash_decoding_static(qd, kvd[:, :Hkv], kvd[:, Hkv:], td, rd, ld, max(lens), o_s, l_s, BS)
        torch.cuda.synchronize()
        assert_o_close(o_s[live.to(DEV)], o_ref[live], "o, own partials, " + what)
        assert_lse_close(l_s, l_ref, "lse, own partials, " + what)
        if nblk >= (max(lens) + 255) // 256:  # (both calls then deal blocks of 256 tokens: the same sums in the same order)
            assert torch.equal(o_s[live.to(DEV)], o_d[live.to(DEV)]) and torch.equal(l_s, l_d), "own partials, " + what


@pytest.mark.parametrize("seed", [3, 11, 42])
def test_random_decode_shapes_on_both_stage1_kernels(lsa, tuning, seed):
    """Seeded random sweep of stage 1 + stage 2 against the oracle, once with the library's own choice of stage-1 kernel
    and once through each shape of the matrix-pipe kernel wherever its conditions hold (plain grid, split waves, listed
    units): ragged batches with requests of a single token,
    of exactly a block, and of a block plus one; groups of 1 to 20 query heads per KV head; blocks of 32 to 512 tokens;
    per-block partials and merged groups of blocks; both dtypes; unused rows and requests in the table."""
    import random
    rng = random.Random(seed)
    for case in range(10):
        dtype = rng.choice([torch.float16, torch.bfloat16])
        Hkv = rng.choice([1, 2, 3, 8])
        group = rng.choice([1, 2, 4, 5, 7, 8, 9, 12, 16, 17, 20])
        Hq = Hkv * group
        BS = rng.choice([32, 64, 96, 128, 256, 384, 512])
        B = rng.choice([1, 2, 5, 9])
        lens = [rng.choice([1, 2, 31, 32, 33, BS - 1, BS, BS + 1, 2 * BS, 3 * BS + 7, 700, 1500, 2600]) for _ in range(B)]
        lens = [max(n, 1) for n in lens]
        merge = rng.choice([1, 1, 2, 4, 16])
        print("case", seed, case, dtype, Hq, Hkv, BS, lens, merge, flush=True)
        D = 128
        q, kv, table, b_req, b_len = decode_case(9000 + 100 * seed + case, B, Hq, Hkv, D, lens, sum(lens) + 200, dtype)
        k, v = kv[:, :Hkv], kv[:, Hkv:]
        o_ref, l_ref = orc.decode_full(q, k, v, table, b_req, b_len)
        kvd, qd, td, rd, ld = kv.to(DEV), q.to(DEV), table.to(DEV), b_req.to(DEV), b_len.to(DEV)
        nblk = (max(lens) + BS - 1) // BS
        for forced in (False, "mfma", "split", "mfma listed"):
            if forced:
                tuning(decode_stage1=forced.split()[0], decode_listed="on" if "listed" in forced else "off")
            else:
                tuning()
            mo_d = torch.full((nblk, B, Hq, D), float("nan"), device=DEV)
            ml_d = torch.full((nblk, B, Hq), float("nan"), device=DEV)
            lsa.longserve_cuda_kernels.flash_decoding_stage1(mo_d, ml_d, qd, kvd[:, :Hkv], kvd[:, Hkv:], td, rd, ld, max(lens), BS, merge)
            o_d = torch.empty(B, Hq, D, device=DEV)
            l_d = torch.empty(B, Hq, device=DEV)
            lsa.longserve_flash_decode_stage2(mo_d, ml_d, ld, o_d, l_d, BS)
            torch.cuda.synchronize()
            what = "seed %d case %d%s" % (seed, case, ", matrix pipe shape " + forced if forced else "")
            reach = torch.tensor([(n + BS - 1) // BS for n in lens])
            untouched = (torch.arange(nblk)[:, None] >= reach[None, :])[:, :, None].expand(nblk, B, Hq)
            assert torch.equal(torch.isnan(ml_d.cpu()), untouched), "rows written, " + what
            assert_o_close(o_d, o_ref, "o, " + what)
            assert_lse_close(l_d, l_ref, "lse, " + what)


@pytest.mark.parametrize("Hq,Hkv,B", [(32, 8, 64), (32, 8, 65), (4, 4, 8), (24, 3, 130), (5, 5, 9)])
def test_equal_shares_at_the_edges_of_their_launches(lsa, tuning, Hq, Hkv, B):
    """Shares forced on batches that are counted in registers (up to 64 requests) and in LDS, merged with one wave and with four
    per (request, head) (up to 1024 pairs), heads that do not fill the merge's groups of four: lengths around the unit of 32
    tokens, empty requests first and last, one request that holds most of the tokens."""
    import random
    rng = random.Random(B)
    tuning(decode_listed="shares")
    lens = [rng.choice([0, 1, 31, 32, 33, 64, 127, 128, 129, 300]) for _ in range(B)]
    lens[0] = lens[-1] = 0
    lens[B // 2] = 5000
    D = 128
    q, kv, table, b_req, b_len = decode_case(300 + B, B, Hq, Hkv, D, lens, sum(lens) + 100, torch.float16)
    o_ref, l_ref = orc.decode_full(q, kv[:, :Hkv], kv[:, Hkv:], table, b_req, b_len)
    kvd = kv.to(DEV)
    nblk = (max(lens) + 255) // 256
    mo_d = torch.full((nblk, B, Hq, D), float("nan"), device=DEV)
    ml_d = torch.full((nblk, B, Hq), float("nan"), device=DEV)
    o_d, l_d = lsa.longserve_token_decode_attention_flash_decoding(q.to(DEV), table.to(DEV), b_req.to(DEV), b_len.to(DEV), mo_d, ml_d, B,
                                                                   max(lens), Hq, D, kvd[:, :Hkv], kvd[:, Hkv:], 256)
    torch.cuda.synchronize()
    assert_o_close(o_d, o_ref, "o")
    assert_lse_close(l_d, l_ref, "lse")


@pytest.mark.parametrize("Hq,Hkv,B,longest,BS", [(32, 8, 128, 200, 256), (32, 8, 256, 256, 256), (32, 32, 65, 130, 256), (32, 8, 128, 1000, 1024)])
def test_batches_of_short_contexts_fill_the_chip(lsa, Hq, Hkv, B, longest, BS):
    """One row of partials per request: right, and in the fused call no slower than three times the two stages called one after
    the other (a few dozen us; dealt as the one share that the rows leave room for, such a batch takes ten to fifty times that)."""
    print("case", Hq, Hkv, B, longest, BS, flush=True)
    D = 128
    lens = [longest - i % 90 for i in range(B)]
    q, kv, table, b_req, b_len = decode_case(700 + B, B, Hq, Hkv, D, lens, sum(lens) + 100, torch.float16)
    o_ref, l_ref = orc.decode_full(q, kv[:, :Hkv], kv[:, Hkv:], table, b_req, b_len)
    qd, kvd, td, rd, ld = q.to(DEV), kv.to(DEV), table.to(DEV), b_req.to(DEV), b_len.to(DEV)
    mo, ml = torch.empty((1, B, Hq, D), device=DEV), torch.empty((1, B, Hq), device=DEV)
    o, l = torch.empty((B, Hq, D), device=DEV), torch.empty((B, Hq), device=DEV)

    def fused():
        lsa.longserve_token_decode_attention_flash_decoding(qd, td, rd, ld, mo, ml, B, longest, Hq, D, kvd[:, :Hkv], kvd[:, Hkv:], BS, o, l)

    def staged():
        lsa.longserve_flash_decode_stage1(qd, kvd[:, :Hkv], kvd[:, Hkv:], td, rd, ld, longest, mo, ml, BS)
        lsa.longserve_flash_decode_stage2(mo, ml, ld, o, l, BS)

    def time_of(call):
        best = math.inf
        for _ in range(4):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(4):
                call()
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b))
        return best

    staged_ms = time_of(staged)
    o.fill_(float("nan"))
    fused_ms = time_of(fused)
    assert_o_close(o, o_ref, "o")
    assert_lse_close(l, l_ref, "lse")
    assert fused_ms < 3 * staged_ms, "%.3f ms fused, %.3f ms in two stages" % (fused_ms, staged_ms)


@pytest.mark.parametrize("shares", [True, False])
def test_fused_call_counts_the_bound_on_lengths_in_whole_blocks(lsa, tuning, shares):
    """max_len_in_batch sizes the launch; a request that is longer within the same 256 tokens is attended to its end, in equal shares
    as on the grids."""
    tuning(decode_listed=None if shares else "off")
    B, Hq, Hkv, D = 24, 32, 8, 128
    lens = [3990, 3905] + [200 + 37 * i for i in range(B - 2)]
    q, kv, table, b_req, b_len = decode_case(41, B, Hq, Hkv, D, lens, sum(lens) + 100, torch.float16)
    o_ref, l_ref = orc.decode_full(q, kv[:, :Hkv], kv[:, Hkv:], table, b_req, b_len)
    kvd = kv.to(DEV)
    mo, ml = torch.empty((16, B, Hq, D), device=DEV), torch.empty((16, B, Hq), device=DEV)
    o, l = lsa.longserve_token_decode_attention_flash_decoding(q.to(DEV), table.to(DEV), b_req.to(DEV), b_len.to(DEV), mo, ml, B, 3900, Hq, D,
                                                               kvd[:, :Hkv], kvd[:, Hkv:], 256)
    assert_o_close(o, o_ref, "o")
    assert_lse_close(l, l_ref, "lse")


def _direct_case(lsa, seed, B, Hq, Hkv, lens, dtype, o_dtype=torch.float32, in_place=False):
    """The fused call and whether it left its partials alone, as the launch does that writes the result itself."""
    D = 128
    q, kv, table, b_req, b_len = decode_case(seed, B, Hq, Hkv, D, lens, sum(lens) + 100, dtype)
    o_ref, l_ref = orc.decode_full(q, kv[:, :Hkv], kv[:, Hkv:], table, b_req, b_len)
    qd, kvd, rows = q.to(DEV), kv.to(DEV), (max(lens) + 255) // 256
    mo, ml = torch.full((rows, B, Hq, D), float("nan"), device=DEV), torch.full((rows, B, Hq), float("nan"), device=DEV)
    o = qd if in_place else torch.full((B, Hq, D), float("nan"), dtype=o_dtype, device=DEV)
    l = torch.full((B, Hq), float("nan"), device=DEV)
    lsa.longserve_token_decode_attention_flash_decoding(qd, table.to(DEV), b_req.to(DEV), b_len.to(DEV), mo, ml, B, max(lens), Hq, D,
                                                        kvd[:, :Hkv], kvd[:, Hkv:], 256, o, l)
    torch.cuda.synchronize()
    # (a result in 16 bits: half a last place of values below 4 on top)
    eps = {torch.float32: 0.0, torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}[o.dtype]
    assert_o_close(o, o_ref, "o", max_abs=O_MAX_ABS + eps, rel=O_REL + eps / 2)
    assert_lse_close(l, l_ref, "lse")
    return bool(torch.isnan(mo).all() and torch.isnan(ml).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("out", ["float32", "same", "other", "in place"])
@pytest.mark.parametrize("Hq,Hkv", [(4, 4), (8, 4), (9, 3), (32, 8), (17, 1), (5, 1)])
def test_short_contexts_in_one_launch(lsa, dtype, out, Hq, Hkv):
    """Lengths around a batch (32), a turn of the four waves (128) and the ends of the range, none among them."""
    print("case", dtype, out, Hq, Hkv, flush=True)
    lens = [0, 1, 31, 32, 33, 0, 127, 128, 129, 160, 161, 255, 256, 257, 319, 320] + ([383, 384] if Hq > Hkv else [])
    other = torch.bfloat16 if dtype == torch.float16 else torch.float16
    assert _direct_case(lsa, 61, len(lens), Hq, Hkv, lens, dtype, {"float32": torch.float32, "other": other}.get(out, dtype), out == "in place")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("BS", [1, 16, 48, 100, 256, 1000])
@pytest.mark.parametrize("rows", [None, 1, 3])
def test_one_launch_attends_the_tokens_that_the_blocks_cover(lsa, tuning, dtype, BS, rows):
    """Any block size, and fewer rows of partials than the longest request fills: the tokens attended are those of the blocks that have a row, as in
    two launches (the fused call's own split kept out by the entry point)."""
    print("case", dtype, BS, rows, flush=True)
    ck, D, B, Hq, Hkv, lens = lsa.longserve_cuda_kernels, 128, 5, 8, 2, [300, 47, 48, 16, 0]
    q, kv, table, b_req, b_len = decode_case(87, B, Hq, Hkv, D, lens, 600, dtype)
    qd, kvd, td, rd, ld = q.to(DEV), kv.to(DEV), table.to(DEV), b_req.to(DEV), b_len.to(DEV)
    n = min(rows or 300, (300 + BS - 1) // BS)
    got = []
    for kernel in (None, "lane"):
        tuning(decode_stage1=kernel)
        mo, ml = torch.full((n, B, Hq, D), float("nan"), device=DEV), torch.full((n, B, Hq), float("nan"), device=DEV)
        o, l = torch.full((B, Hq, D), float("nan"), device=DEV), torch.full((B, Hq), float("nan"), device=DEV)
        if kernel:  # two launches; the merge reads the rows there are
            ck.flash_decoding_stage1(mo, ml, qd, kvd[:, :Hkv], kvd[:, Hkv:], td, rd, ld, 300, BS)
            ck.flash_decoding_stage2(o, l, torch.clamp(ld, max=n * BS), mo, ml, BS)
        else:
            ck.flash_decoding(mo, ml, qd, kvd[:, :Hkv], kvd[:, Hkv:], td, rd, ld, 300, o, l, BS)
        torch.cuda.synchronize()
        assert bool(torch.isnan(mo).all()) == (kernel is None)
        got.append((o.cpu(), l.cpu()))
    (o, l), (o2, l2) = got
    o_ref, l_ref = orc.decode_full(q, kv[:, :Hkv], kv[:, Hkv:], table, b_req, torch.clamp(b_len, max=n * BS))
    for x, y, what in ((o, o2, "o against two launches"), (o, o_ref, "o")):
        assert_o_close(x, y, what)
    assert_lse_close(l, l2, "lse against two launches")
    assert_lse_close(l, l_ref, "lse")


def _kernel_nodes(graph):
    """How many nodes a captured graph has."""
    import ctypes
    n = ctypes.c_size_t()
    hip = ctypes.CDLL("libamdhip64.so")
    assert hip.hipGraphGetNodes(ctypes.c_void_p(int(graph.raw_cuda_graph())), None, ctypes.byref(n)) == 0
    return n.value


# per request at most 3 partials; the most that one of four, eight, five heads, of one, two and three in the lane kernel take (128 and 64 rows); one more
@pytest.mark.parametrize("Hq,Hkv,lens,joined", [
    (32, 8, [0, 1, 255, 256, 257, 0, 511, 513, 700, 768], True), (8, 2, [8192], True), (8, 2, [8193], False), (8, 1, [2048, 300, 5], True), (8, 1, [2049], False),
    (5, 1, [3072, 1, 0], True), (4, 4, [16384], True), (4, 4, [16385], False), (8, 4, [8192, 256, 257], True), (8, 4, [8193], False),
    (9, 3, [5376, 31, 129], True), (3, 1, [5377], False), (9, 1, [600], False), (17, 1, [600], False), (16, 8, [385, 0, 2000], True),
    (32, 8, [2048] * 8, True), (32, 8, [8192, 700], False)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("out", ["float32", "same", "other"])
def test_partials_merged_in_the_launch_that_wrote_them(lsa, Hq, Hkv, lens, joined, dtype, out):
    """The last workgroup on a request merges its partials, whatever the result's memory held before (where the workgroups count each
    other); replayed from a graph among other calls over the same memory it counts anew every time."""
    print("case", Hq, Hkv, lens[:3], dtype, out, flush=True)
    B, D = len(lens), 128
    q, kv, table, b_req, b_len = decode_case(93, B, Hq, Hkv, D, lens, sum(lens) + 100, dtype)
    o_ref, l_ref = orc.decode_full(q, kv[:, :Hkv], kv[:, Hkv:], table, b_req, b_len)
    qd, kvd, td, rd, ld, rows = q.to(DEV), kv.to(DEV), table.to(DEV), b_req.to(DEV), b_len.to(DEV), (max(lens) + 255) // 256
    mo, ml = torch.full((rows, B, Hq, D), float("nan"), device=DEV), torch.full((rows, B, Hq), float("nan"), device=DEV)
    other = torch.bfloat16 if dtype == torch.float16 else torch.float16
    o = torch.empty((B, Hq, D), dtype={"float32": torch.float32, "other": other}.get(out, dtype), device=DEV)
    l = torch.empty((B, Hq), device=DEV)
    words = o.view(torch.int64)

    def call():
        lsa.longserve_token_decode_attention_flash_decoding(qd, td, rd, ld, mo, ml, B, max(lens), Hq, D, kvd[:, :Hkv], kvd[:, Hkv:], 256, o, l)

    # (a result in 16 bits: half a last place of values below 4 on top)
    eps = {torch.float32: 0.0, torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}[o.dtype]
    first = None
    for held in (0, -1, 1, 2, 0x7fffffffffffffff, -2 ** 63, None):  # (None: the last call's result)
        if held is not None:
            words.fill_(held)
        call()
        torch.cuda.synchronize()
        if first is None:
            first = (o.clone(), l.clone())
            assert_o_close(o, o_ref, "o", max_abs=O_MAX_ABS + eps, rel=O_REL + eps / 2)
            assert_lse_close(l, l_ref, "lse")
        assert torch.equal(o, first[0]) and torch.equal(l, first[1]), held
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        call()
    assert (_kernel_nodes(graph) == 1) == joined
    q2 = torch.roll(qd, 1, 1)
    for turn in range(4):
        o.view(torch.uint8).random_(0, 256)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(o, first[0]) and torch.equal(l, first[1]), turn
        if turn == 1:  # other eager work over the same result and partials
            keep = qd.clone()
            qd.copy_(q2)
            call()
            qd.copy_(keep)


@pytest.mark.parametrize("Hq,Hkv,B,longest,direct", [
    (4, 4, 1, 320, True), (4, 4, 1, 321, False), (4, 4, 127, 20, True), (4, 4, 128, 20, False), (8, 4, 255, 30, True), (8, 4, 256, 30, False),
    (8, 4, 1, 384, True), (8, 4, 1, 385, False), (8, 4, 64, 385, False), (32, 8, 300, 40, False), (32, 8, 256, 40, True), (32, 8, 31, 385, False),
    (32, 8, 31, 384, True), (32, 8, 32, 640, True), (32, 8, 32, 641, False), (8, 1, 256, 640, True), (8, 1, 2049, 30, True),
    (8, 1, 256, 1024, False), (32, 8, 48, 1024, False), (32, 8, 64, 800, False), (32, 8, 16, 512, False), (16, 8, 48, 512, False)])
def test_which_short_contexts_take_one_launch(lsa, Hq, Hkv, B, longest, direct):
    """One long request among short ones, for which one launch is no faster than a walk of the long one: past 640 tokens, and past 384 on part
    of the CUs, two launches share it (48 requests on 32/8 heads, one of 1024 tokens, 15.0 us in two, 20.3 in one)."""
    print("case", Hq, Hkv, B, longest, flush=True)
    assert _direct_case(lsa, 67, B, Hq, Hkv, [longest] + [1 + (7 * i) % min(longest, 60) for i in range(B - 1)], torch.bfloat16) == direct


def test_result_over_the_queries_takes_two_launches(lsa):
    """A result that lies over the queries row for row is written in one launch; shifted against them it waits for the last read."""
    B, Hq, Hkv, D = 6, 8, 2, 128
    lens = [100, 1, 300, 64, 256, 31]
    q, kv, table, b_req, b_len = decode_case(71, B, Hq, Hkv, D, lens, 1000, torch.float16)
    o_ref, l_ref = orc.decode_full(q, kv[:, :Hkv], kv[:, Hkv:], table, b_req, b_len)
    kvd = kv.to(DEV)
    for shift, direct in ((0, True), (D, False), (B * Hq * D, True)):
        room = torch.zeros(2 * B * Hq * D, dtype=torch.float16, device=DEV)
        qd, o = room[shift:shift + B * Hq * D].view(B, Hq, D), room[:B * Hq * D].view(B, Hq, D)
        qd.copy_(q)
        mo, ml = torch.full((2, B, Hq, D), float("nan"), device=DEV), torch.empty((2, B, Hq), device=DEV)
        l = torch.empty((B, Hq), device=DEV)
        lsa.longserve_token_decode_attention_flash_decoding(qd, table.to(DEV), b_req.to(DEV), b_len.to(DEV), mo, ml, B, 300, Hq, D,
                                                            kvd[:, :Hkv], kvd[:, Hkv:], 256, o, l)
        assert bool(torch.isnan(mo).all()) == direct
        assert_o_close(o, o_ref, "o", max_abs=O_MAX_ABS + 2.0 ** -10, rel=O_REL + 2.0 ** -11)
        assert_lse_close(l, l_ref, "lse")


@pytest.mark.parametrize("call", ["native", "checked", "static"])
@pytest.mark.parametrize("where", ["apart", "o over K", "o over V", "o over the table", "lse over K", "lse over the table"])
def test_result_over_the_pool_or_the_table_is_written_behind_the_last_read(lsa, monkeypatch, call, where):
    """Short contexts whose result lies over rows of the pool, or of the table, that requests still read: two launches, as for calls of the C ABI that do
    not say that it lies apart."""
    print("case", call, where, flush=True)
    ck, D, B, Hq, Hkv, lens = lsa.longserve_cuda_kernels, 128, 8, 8, 2, [100, 1, 300, 64, 256, 31, 200, 128]
    if call == "checked":
        monkeypatch.setattr(ck._native, "token_decode_attention", lambda *a: None)
    q, kv, table, b_req, b_len = decode_case(83, B, Hq, Hkv, D, lens, 2000, torch.float16, pad_seq=200)
    o_ref, l_ref = orc.decode_full(q, kv[:, :Hkv], kv[:, Hkv:], table, b_req, b_len)
    qd, rd, ld, td = q.to(DEV), b_req.to(DEV), b_len.to(DEV), table.to(DEV).contiguous()
    pool = torch.cat([kv[:, :Hkv].reshape(-1), kv[:, Hkv:].reshape(-1)]).to(DEV)  # (K and V apart, so that either can be met alone)
    k, v = pool[:pool.numel() // 2].view(-1, Hkv, D), pool[pool.numel() // 2:].view(-1, Hkv, D)
    n = B * Hq * D
    o = {"o over K": k.reshape(-1)[:n], "o over V": v.reshape(-1)[n:2 * n], "o over the table": td.view(-1)[:n // 2].view(torch.float16)}.get(
        where, torch.zeros(n, dtype=torch.float16, device=DEV))
    l = {"lse over K": k.reshape(-1)[:2 * B * Hq].view(torch.float32), "lse over the table": td.view(-1)[:B * Hq].view(torch.float32)}.get(
        where, torch.zeros(B * Hq, device=DEV))
    o, l = o.view(B, Hq, D), l.view(B, Hq)
    mo, ml = torch.full((2, B, Hq, D), float("nan"), device=DEV), torch.full((2, B, Hq), float("nan"), device=DEV)
    if call == "static":
        ck.flash_decoding_static(qd, k, v, td, rd, ld, max(lens), o, l, 256)
    else:
        ck.flash_decoding(mo, ml, qd, k, v, td, rd, ld, max(lens), o, l, 256)
        assert bool(torch.isnan(mo).all()) == (where == "apart")
    torch.cuda.synchronize()
    assert_o_close(o, o_ref, "o", max_abs=O_MAX_ABS + 2.0 ** -10, rel=O_REL + 2.0 ** -11)
    assert_lse_close(l, l_ref, "lse")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_one_launch_and_infinite_keys_and_values(lsa, tuning, dtype):
    """Scores of minus infinity weigh nothing (a request of nothing else has the result of an empty one) and infinite values stay
    infinite, as in the lane kernel's two launches."""
    B, H, D = 5, 4, 128
    lens = [32, 40, 200, 129, 64]
    q, kv, table, b_req, b_len = decode_case(73, B, H, H, D, lens, 600, dtype)
    q = q.abs() + 0.125
    slot = [table[int(b_req[b])] for b in range(B)]
    kv[slot[0][:32].long(), :H] = float("-inf")                # nothing but -inf
    kv[slot[1][:32].long(), :H] = float("-inf")                # the first batch
    kv[slot[2][130:200].long(), :H] = float("-inf")            # whole waves at the end
    kv[slot[3][7].long(), H:, 5] = float("inf")
    kv[slot[3][90].long(), H:, 6] = float("-inf")
    qd, kvd = q.to(DEV), kv.to(DEV)
    got = []
    for kernel in (None, "lane"):
        tuning(decode_stage1=kernel)
        mo, ml = torch.full((1, B, H, D), float("nan"), device=DEV), torch.full((1, B, H), float("nan"), device=DEV)
        o, l = lsa.longserve_token_decode_attention_flash_decoding(qd, table.to(DEV), b_req.to(DEV), b_len.to(DEV), mo, ml, B, 200, H, D,
                                                                   kvd[:, :H], kvd[:, H:], 256)
        torch.cuda.synchronize()
        assert bool(torch.isnan(mo).all()) == (kernel is None)
        got.append((o.cpu(), l.cpu()))
    (o, l), (o2, l2) = got
    assert torch.equal(o.isinf() * o.sign(), o2.isinf() * o2.sign()) and torch.equal(o.isnan(), o2.isnan())
    fin = o2.isfinite()
    assert_o_close(o[fin], o2[fin], "o")
    assert_lse_close(l, l2, "lse")


@pytest.mark.parametrize("dtype,huge", [(torch.float16, 65504.0), (torch.bfloat16, 3e38)])
@pytest.mark.parametrize("Hq,Hkv", [(4, 4), (8, 2)])
def test_one_launch_and_huge_values_that_weigh_nothing(lsa, dtype, huge, Hq, Hkv):
    """Tokens with scores of minus infinity and values at the end of the type's range, among them the last one, which the places past a request's end
    repeat: the sum over the others, small by comparison, is as if they were not there."""
    print("case", dtype, Hq, Hkv, flush=True)
    D, lens = 128, [33, 40, 200, 129, 1 + 128 + 31]
    q, kv, table, b_req, b_len = decode_case(79, len(lens), Hq, Hkv, D, lens, 700, dtype)
    q = q.abs() + 0.125
    kv[:, Hkv:] = kv[:, Hkv:] * 2.0 ** -10
    for b, n in enumerate(lens):
        gone = table[int(b_req[b])][[0, n // 2, n - 1]].long()
        kv[gone, :Hkv] = float("-inf")
        kv[gone, Hkv:] = huge
    o_ref, l_ref = orc.decode_full(q, kv[:, :Hkv], kv[:, Hkv:], table, b_req, b_len)
    kvd = kv.to(DEV)
    mo, ml = torch.full((1, len(lens), Hq, D), float("nan"), device=DEV), torch.full((1, len(lens), Hq), float("nan"), device=DEV)
    o, l = lsa.longserve_token_decode_attention_flash_decoding(q.to(DEV), table.to(DEV), b_req.to(DEV), b_len.to(DEV), mo, ml, len(lens), max(lens), Hq, D,
                                                               kvd[:, :Hkv], kvd[:, Hkv:], 256)
    torch.cuda.synchronize()
    assert bool(torch.isnan(mo).all())  # (one launch)
    # (2^-10 of what the sums of values around 1 are held to)
    assert_o_close(o * 2.0 ** 10, o_ref * 2.0 ** 10, "o")
    assert_lse_close(l, l_ref, "lse")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Hq,Hkv,lens", [
    (32, 8, [32769]), (32, 8, [33000]), (64, 8, [17000, 33]), (32, 32, [8193]),  # one request and two, merged by sixteen waves a pair (64 pairs)
    (32, 4, [20000, 0, 17001]), (32, 8, [9000, 1, 33, 8999]),                    # more pairs, a request without tokens
    (8, 1, [70000, 1, 300, 69999]), (16, 1, [33819] + [2000] * 7),               # one KV head, 1096 and 1064 waves
    (4, 1, [131400, 500, 131072, 64]),                                           # ... and 2056
    (32, 8, [592, 576] + [40] * 22, ), (32, 4, [36 * 256 - 100, 7, 2000, 1]),    # 576 waves: the shape whose waves split a block
])
def test_launches_of_a_few_workgroups_past_a_round(lsa, dtype, Hq, Hkv, lens):
    """Few requests in equal shares, and the last launch that is split among a block's waves, as the library chooses."""
    print("case", dtype, Hq, Hkv, lens[:4], flush=True)
    B, D, BS = len(lens), 128, 256
    q, kv, table, b_req, b_len = decode_case(321, B, Hq, Hkv, D, lens, sum(lens) + 500, dtype)
    o_ref, l_ref = orc.decode_full(q, kv[:, :Hkv], kv[:, Hkv:], table, b_req, b_len)
    kvd = kv.to(DEV)
    mo = torch.full((max(lens) // BS + 1, B, Hq, D), float("nan"), device=DEV)
    ml = torch.full(mo.shape[:3], float("nan"), device=DEV)
    for _ in range(2):  # (the second call over what the first left in the buffers)
        o, l = lsa.longserve_token_decode_attention_flash_decoding(q.to(DEV), table.to(DEV), b_req.to(DEV), b_len.to(DEV), mo, ml, B, max(lens), Hq, D,
                                                                   kvd[:, :Hkv], kvd[:, Hkv:], BS)
        torch.cuda.synchronize()
        live = b_len > 0
        assert_o_close(o.cpu()[live], o_ref[live], "o")
        assert_lse_close(l.cpu()[live], l_ref[live], "lse")
        assert bool((o.cpu()[~live] == 0).all()) and bool((l.cpu()[~live] == -math.inf).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Hq,Hkv,lens", [(32, 8, [32 * 256 + 1, 300, 0, 4000]), (16, 8, [48 * 256, 7, 2000, 12287]), (32, 32, [3072, 1, 3000, 257])])
def test_both_stages_of_launches_just_past_a_workgroup_per_cu(lsa, dtype, Hq, Hkv, lens):
    """1056 to 1536 waves, split among a block's waves: the stages apart, one partial per 256 tokens, in buffers that start as NaN."""
    print("case", dtype, Hq, Hkv, lens, flush=True)
    B, D, BS = len(lens), 128, 256
    q, kv, table, b_req, b_len = decode_case(77, B, Hq, Hkv, D, lens, sum(lens) + 500, dtype)
    o_ref, l_ref = orc.decode_full(q, kv[:, :Hkv], kv[:, Hkv:], table, b_req, b_len)
    kvd = kv.to(DEV)
    nblk = (max(lens) + BS - 1) // BS
    mo, ml = torch.full((nblk, B, Hq, D), float("nan"), device=DEV), torch.full((nblk, B, Hq), float("nan"), device=DEV)
    o, l = torch.empty(B, Hq, D, device=DEV), torch.empty(B, Hq, device=DEV)
    lsa.longserve_flash_decode_stage1(q.to(DEV), kvd[:, :Hkv], kvd[:, Hkv:], table.to(DEV), b_req.to(DEV), b_len.to(DEV), max(lens), mo, ml, BS)
    lsa.longserve_flash_decode_stage2(mo, ml, b_len.to(DEV), o, l, BS)
    torch.cuda.synchronize()
    written = torch.arange(nblk)[:, None] * BS < b_len[None, :]
    assert torch.equal(~torch.isnan(ml.cpu()), written[:, :, None].expand(-1, -1, Hq))
    live = b_len > 0
    assert_o_close(o.cpu()[live], o_ref[live], "o")
    assert_lse_close(l.cpu()[live], l_ref[live], "lse")


def _against_64_bits(o, q, kv, table, b_req, lens, Hkv):
    """Relative error of the decode result o against the same in 64 bits, over all requests and heads."""
    off = norm = 0.0
    for b, n in enumerate(lens):
        rows = kv[table[b_req[b].long(), :n].long()]
        for h in range(q.shape[1]):
            kvh = h * Hkv // q.shape[1]
            w = torch.softmax(rows[:, kvh].double() @ q[b, h].double() / math.sqrt(128), 0)
            ref = w @ rows[:, Hkv + kvh].double()
            off += float((o[b, h].double() - ref).square().sum())
            norm += float(ref.square().sum())
    return math.sqrt(off / norm)


@pytest.mark.parametrize("Hq,Hkv,lens,BS", [(1, 1, [131870] * 2, 256), (3, 1, [87914, 87914, 300], 256), (2, 1, [65936] * 4, 256), (10, 5, [65936], 256),
                                            (32, 32, [16384], 1024), (16, 4, [60000] * 2, 1056)])
def test_long_contexts_in_bf16_keep_the_weights_in_full(lsa, Hq, Hkv, lens, BS):
    """Few coarse blocks of contexts long enough for equal shares: the weights that multiply V stay fp32.  In two bf16 parts they have 16 bits, a rounding of
    2^-17 / sqrt(3) = 4.4e-6 each, and the result's relative error is that of its weights; in full what is left are fp32's own roundings, below a tenth of that."""
    print("case", Hq, Hkv, lens, BS, flush=True)
    B, D = len(lens), 128
    g = torch.Generator(device=DEV).manual_seed(5)
    q = torch.empty(B, Hq, D, dtype=torch.bfloat16, device=DEV).normal_(0.0, 0.5, generator=g)
    kv = torch.empty(sum(lens) + 100, 2 * Hkv, D, dtype=torch.bfloat16, device=DEV).normal_(0.0, 0.5, generator=g)
    slots = torch.randperm(kv.shape[0], generator=g, device=DEV).int()
    table, at = torch.zeros(B, max(lens), dtype=torch.int32, device=DEV), 0
    for b, n in enumerate(lens):
        table[b, :n] = slots[at:at + n]
        at += n
    b_len, b_req = torch.tensor(lens, dtype=torch.int32, device=DEV), torch.arange(B, dtype=torch.int32, device=DEV)
    mo = torch.empty(max(lens) // BS + 1, B, Hq, D, device=DEV)
    ml = torch.empty(mo.shape[:3], device=DEV)
    o, _ = lsa.longserve_token_decode_attention_flash_decoding(q, table, b_req, b_len, mo, ml, B, max(lens), Hq, D, kv[:, :Hkv], kv[:, Hkv:], BS)
    torch.cuda.synchronize()
    assert _against_64_bits(o, q, kv, table, b_req, lens, Hkv) < 2.0 ** -19


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Hq,Hkv,lens", [(16, 16, [3328, 900, 2000, 40, 2700]), (32, 32, [8448]), (32, 8, [33 * 256, 300, 0, 4000])])
def test_stage1_just_past_a_workgroup_per_cu_runs_the_plain_shape(lsa, tuning, dtype, Hq, Hkv, lens):
    """1040 to 1056 waves, where the shape whose waves split a block takes up to a fifth longer: the partials are the plain shape's, bit for bit."""
    print("case", dtype, Hq, Hkv, lens, flush=True)
    B, BS = len(lens), 256
    q, kv, table, b_req, b_len = decode_case(78, B, Hq, Hkv, 128, lens, sum(lens) + 500, dtype)
    qd, kvd, td, rd, ld = q.to(DEV), kv.to(DEV), table.to(DEV), b_req.to(DEV), b_len.to(DEV)
    nblk = (max(lens) + BS - 1) // BS

    def partials():
        mo, ml = torch.zeros((nblk, B, Hq, 128), device=DEV), torch.zeros((nblk, B, Hq), device=DEV)
        lsa.longserve_flash_decode_stage1(qd, kvd[:, :Hkv], kvd[:, Hkv:], td, rd, ld, max(lens), mo, ml, BS)
        torch.cuda.synchronize()
        return mo, ml

    got = partials()
    tuning(decode_stage1="mfma")
    want = partials()
    tuning(decode_stage1="split")
    other = partials()
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    assert not torch.equal(other[0], want[0])  # (the two shapes can be told apart)


@pytest.mark.parametrize("Hq,Hkv,lens,shares", [
    (16, 16, [10240] * 3, False), (32, 8, [8961, 300, 7000, 6453], False), (32, 8, [10752] * 4, False), (32, 8, [10753, 9000, 40, 10000], True), (32, 8, [12288] * 4, True), (32, 8, [12289] * 4, False), (32, 8, [15000, 300, 4000], False),
    (32, 8, [32768], False), (32, 8, [33023], False), (32, 8, [33024], True), (32, 8, [57344], True), (32, 8, [57600], False), (32, 8, [65537], False), (32, 8, [65792], True),
    (16, 16, [24576], True), (16, 16, [24832], False), (16, 16, [33024], True), (16, 16, [53248], True), (16, 16, [53504], False), (16, 16, [65792], True)])
def test_few_requests_in_equal_shares_where_these_are_no_slower(lsa, Hq, Hkv, lens, shares):
    """A grid leaves one partial per block of a request; equal shares leave others.  On both sides of every line of the rule."""
    from loongserve_amd.decoding import _fused_block_seq
    print("case", Hq, Hkv, lens, flush=True)
    B, D, BS = len(lens), 128, 256
    q, kv, table, b_req, b_len = decode_case(322, B, Hq, Hkv, D, lens, sum(lens) + 500, torch.float16)
    o_ref, l_ref = orc.decode_full(q, kv[:, :Hkv], kv[:, Hkv:], table, b_req, b_len)
    kvd = kv.to(DEV)
    mo = torch.full((max(lens) // BS + 1, B, Hq, D), float("nan"), device=DEV)
    ml = torch.full(mo.shape[:3], float("nan"), device=DEV)
    o, l = lsa.longserve_token_decode_attention_flash_decoding(q.to(DEV), table.to(DEV), b_req.to(DEV), b_len.to(DEV), mo, ml, B, max(lens), Hq, D,
                                                               kvd[:, :Hkv], kvd[:, Hkv:], BS)
    torch.cuda.synchronize()
    assert_o_close(o, o_ref, "o")
    assert_lse_close(l, l_ref, "lse")
    split = _fused_block_seq(BS, B, max(lens), Hkv)
    blocks = sum(-(-n // split) for n in lens) * Hq
    assert (int((~ml.isnan()).sum()) != blocks) == shares


@pytest.mark.parametrize("Hq,Hkv,lens,shares", [
    (16, 1, [61952, 30000, 200, 5000, 100], False), (8, 1, [34000] + [700] * 7, False), (8, 1, [16640] + [700] * 15, False), (8, 1, [11264] + [700] * 23, True), (8, 1, [13568] + [5000] * 23, True), (8, 1, [13569] + [700] * 23, False),
    (8, 1, [6400] + [50] * 83, True), (8, 1, [6144] + [50] * 95, True), (8, 1, [6145] + [50] * 95, False), (8, 1, [175360, 300, 7000], False), (8, 1, [3000] + [50] * 99, True), (8, 1, [2800] + [50] * 100, False), (12, 3, [64000, 4000, 6133], False)])
def test_few_kv_heads_in_equal_shares_where_these_are_no_slower(lsa, Hq, Hkv, lens, shares):
    """As above for fewer than four KV heads, against the shape whose waves split a block."""
    test_few_requests_in_equal_shares_where_these_are_no_slower(lsa, Hq, Hkv, lens, shares)


@pytest.mark.parametrize("Hq,Hkv,lens,block,joined", [
    (8, 1, [768] * 30, 1024, False), (8, 2, [770] * 64, 256, True), (8, 2, [513] * 86, 256, False),  # one partial; 512 and 516 workgroups
    (8, 2, [4000] * 8, 256, True), (8, 2, [4097] * 8, 256, False), (4, 1, [8190] * 30, 1024, True), (4, 1, [8190] * 33, 1024, False), (4, 1, [4090] * 33, 512, True),  # 64 and 68 rows; 240 and 264 workgroups
    (8, 4, [2000, 5], 128, True), (4, 4, [1500], 128, True), (8, 2, [1025, 0, 300], 128, True)])  # one and two heads of the lane kernel, four: several blocks per 256 tokens
def test_partials_are_merged_in_their_launch_where_that_is_no_slower(lsa, Hq, Hkv, lens, block, joined):
    """A graph of the fused call is one kernel or two, by the workgroups, the block and the partials, and either gives the result again and again."""
    print("case", Hq, Hkv, lens[:2], len(lens), block, flush=True)
    B, D = len(lens), 128
    q, kv, table, b_req, b_len = decode_case(97, B, Hq, Hkv, D, lens, sum(lens) + 100, torch.float16)
    o_ref, l_ref = orc.decode_full(q, kv[:, :Hkv], kv[:, Hkv:], table, b_req, b_len)
    qd, kvd, td, rd, ld, rows = q.to(DEV), kv.to(DEV), table.to(DEV), b_req.to(DEV), b_len.to(DEV), (max(lens) + block - 1) // block
    mo, ml = torch.full((rows, B, Hq, D), float("nan"), device=DEV), torch.full((rows, B, Hq), float("nan"), device=DEV)
    o, l = torch.empty((B, Hq, D), device=DEV), torch.empty((B, Hq), device=DEV)

    def call():
        lsa.longserve_cuda_kernels.flash_decoding(mo, ml, qd, kvd[:, :Hkv], kvd[:, Hkv:], td, rd, ld, max(lens), o, l, block)

    call()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        call()
    assert (_kernel_nodes(graph) == 1) == joined
    graph.instantiate()
    for held in (0, -1, None):
        if held is not None:
            o.view(torch.int64).fill_(held)
        graph.replay()
        torch.cuda.synchronize()
        assert_o_close(o, o_ref, "o")
        assert_lse_close(l, l_ref, "lse")


def _kernel_threads(graph):
    """The threads per workgroup of a captured graph's kernels, in no order."""
    import ctypes

    class Params(ctypes.Structure):  # hipKernelNodeParams
        _fields_ = [("block", ctypes.c_uint * 3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("grid", ctypes.c_uint * 3),
                    ("args", ctypes.c_void_p), ("lds", ctypes.c_uint)]

    hip, n = ctypes.CDLL("libamdhip64.so"), ctypes.c_size_t(_kernel_nodes(graph))
    nodes, found = (ctypes.c_void_p * n.value)(), []
    assert hip.hipGraphGetNodes(ctypes.c_void_p(int(graph.raw_cuda_graph())), nodes, ctypes.byref(n)) == 0
    for node in nodes:
        p = Params()
        assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(p)) == 0
        found.append(p.block[0] * p.block[1] * p.block[2])
    return sorted(found)


@pytest.mark.parametrize("Hq,Hkv,lens,threads", [(4, 4, [70000], 1024), (32, 8, [33000, 300], 1024), (8, 8, [5000] + [600] * 7, 256), (4, 4, [5120] + [300] * 15, 256)])
def test_shares_of_many_requests_are_merged_by_four_waves(lsa, Hq, Hkv, lens, threads):
    """Sixteen waves a (request, head) pair for one or two requests, whose rows are many; up to 64 pairs of more requests have few each."""
    print("case", Hq, Hkv, lens[:2], flush=True)
    B, D, BS = len(lens), 128, 256
    q, kv, table, b_req, b_len = decode_case(323, B, Hq, Hkv, D, lens, sum(lens) + 500, torch.float16)
    o_ref, l_ref = orc.decode_full(q, kv[:, :Hkv], kv[:, Hkv:], table, b_req, b_len)
    qd, kvd, td, rd, ld = q.to(DEV), kv.to(DEV), table.to(DEV), b_req.to(DEV), b_len.to(DEV)
    mo = torch.full((max(lens) // BS + 1, B, Hq, D), float("nan"), device=DEV)
    ml = torch.full(mo.shape[:3], float("nan"), device=DEV)
    o, l = torch.empty((B, Hq, D), device=DEV), torch.empty((B, Hq), device=DEV)
    call = lambda: lsa.longserve_token_decode_attention_flash_decoding(qd, td, rd, ld, mo, ml, B, max(lens), Hq, D, kvd[:, :Hkv], kvd[:, Hkv:], BS, o, l)
    call()
    torch.cuda.synchronize()
    assert_o_close(o, o_ref, "o")
    assert_lse_close(l, l_ref, "lse")
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        call()
    assert _kernel_threads(graph) == sorted([256, threads])


@pytest.mark.parametrize("lens,shape", [([17408], "split"), ([17409], "mfma"), ([1281] * 12, "mfma"), ([4352, 7, 900, 3000], "split")])
def test_stage1_is_split_among_a_blocks_waves_up_to_544_waves(lsa, tuning, lens, shape):
    """On 32/8 heads: above that a batch of one length takes longer than in the plain shape.  The partials tell which of the two ran."""
    print("case", lens[:2], flush=True)
    B, BS = len(lens), 256
    q, kv, table, b_req, b_len = decode_case(79, B, 32, 8, 128, lens, sum(lens) + 500, torch.float16)
    qd, kvd, td, rd, ld = q.to(DEV), kv.to(DEV), table.to(DEV), b_req.to(DEV), b_len.to(DEV)
    nblk = (max(lens) + BS - 1) // BS
    got = {}
    for how in (None, "split", "mfma"):
        tuning(decode_stage1=how)
        got[how] = torch.zeros((nblk, B, 32, 128), device=DEV)
        ml = torch.zeros((nblk, B, 32), device=DEV)
        lsa.longserve_flash_decode_stage1(qd, kvd[:, :8], kvd[:, 8:], td, rd, ld, max(lens), got[how], ml, BS)
    torch.cuda.synchronize()
    assert torch.equal(got[None], got[shape]) and not torch.equal(got["split"], got["mfma"])


def _managed(shape):
    """A float32 tensor of this GPU over managed memory, which is not freed."""
    import ctypes
    hip, ptr, n = ctypes.CDLL("libamdhip64.so"), ctypes.c_void_p(), math.prod(shape)
    assert hip.hipMallocManaged(ctypes.byref(ptr), ctypes.c_size_t(4 * n), ctypes.c_uint(1)) == 0
    t = torch.as_tensor(type("Held", (), {"__cuda_array_interface__": dict(shape=tuple(shape), typestr="<f4", data=(ptr.value, False), version=2)})(), device=DEV)
    assert t.data_ptr() == ptr.value and t.is_cuda
    return t


@pytest.mark.parametrize("static", [False, True])
def test_results_in_other_memory_than_the_gpus_own_take_two_launches(lsa, static):
    """Workgroups count each other in the result only where the runtime knows it as the GPU's own memory; a tensor over managed memory is written behind
    the last read, by two launches, whichever call it is handed to."""
    lens, Hq, Hkv, D = [1500, 700], 32, 8, 128
    q, kv, table, b_req, b_len = decode_case(98, 2, Hq, Hkv, D, lens, 3000, torch.float16)
    o_ref, l_ref = orc.decode_full(q, kv[:, :Hkv], kv[:, Hkv:], table, b_req, b_len)
    qd, kvd, td, rd, ld = q.to(DEV), kv.to(DEV), table.to(DEV), b_req.to(DEV), b_len.to(DEV)
    mo, ml = torch.empty((6, 2, Hq, D), device=DEV), torch.empty((6, 2, Hq), device=DEV)
    for o, kernels in ((torch.empty((2, Hq, D), device=DEV), 1), (_managed((2, Hq, D)), 2)):
        l = torch.empty((2, Hq), device=DEV)

        def call():
            if static:
                lsa.longserve_cuda_kernels.flash_decoding_static(qd, kvd[:, :Hkv], kvd[:, Hkv:], td, rd, ld, max(lens), o, l, 256)
            else:
                lsa.longserve_token_decode_attention_flash_decoding(qd, td, rd, ld, mo, ml, 2, max(lens), Hq, D, kvd[:, :Hkv], kvd[:, Hkv:], 256, o, l)

        graph = torch.cuda.CUDAGraph(keep_graph=True)
        with torch.cuda.graph(graph):
            call()
        assert _kernel_nodes(graph) == kernels
        o.fill_(float("nan"))
        call()
        torch.cuda.synchronize()
        assert_o_close(o, o_ref, "o")
        assert_lse_close(l, l_ref, "lse")


@pytest.mark.parametrize("lead", [7, 2 ** 62, 2 ** 63 - 1])
def test_stage2_with_more_rows_of_peers_than_there_are(lsa, lead):
    """Every row of the buffer is merged, whatever the length is, as for lead_rows of all its rows."""
    print("case", lead, flush=True)
    g = torch.Generator().manual_seed(3)
    mo, ml = torch.randn(7, 3, 2, 128, generator=g).to(DEV), torch.randn(7, 3, 2, generator=g).to(DEV)
    w = torch.softmax(ml.double(), 0)
    want, want_lse = (w[..., None] * mo.double()).sum(0).float(), torch.logsumexp(ml.double(), 0).float()
    for lens in ([0, 1, 5], [2 ** 31 - 1] * 3):
        o, l = torch.zeros((3, 2, 128), device=DEV), torch.zeros((3, 2), device=DEV)
        lsa.longserve_flash_decode_stage2(mo, ml, torch.tensor(lens, dtype=torch.int32, device=DEV), o, l, 1, lead)
        torch.cuda.synchronize()
        assert_o_close(o.cpu(), want.cpu(), "o")
        assert_lse_close(l.cpu(), want_lse.cpu(), "lse", rel=1e-5)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Hq,Hkv,lens,BS", [(3, 1, [131870, 300], 256), (10, 5, [65936], 256), (16, 4, [60000, 7], 1056)])
def test_long_contexts_of_few_coarse_blocks_run_the_lane_kernel(lsa, tuning, dtype, Hq, Hkv, lens, BS):
    """Whose weights are rounded least: the bits are those of the forced choice."""
    print("case", dtype, Hq, Hkv, lens, BS, flush=True)
    B = len(lens)
    q, kv, table, b_req, b_len = decode_case(80, B, Hq, Hkv, 128, lens, sum(lens) + 100, dtype)
    qd, kvd, td, rd, ld = q.to(DEV), kv.to(DEV), table.to(DEV), b_req.to(DEV), b_len.to(DEV)
    got = []
    for how in (None, "lane"):
        tuning(decode_stage1=how)
        mo = torch.empty(max(lens) // BS + 1, B, Hq, 128, device=DEV)
        ml = torch.empty(mo.shape[:3], device=DEV)
        got.append(lsa.longserve_token_decode_attention_flash_decoding(qd, td, rd, ld, mo, ml, B, max(lens), Hq, 128, kvd[:, :Hkv], kvd[:, Hkv:], BS))
    torch.cuda.synchronize()
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
