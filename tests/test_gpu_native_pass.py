"""The operators' native argument pass (csrc/binding.cpp) beside the checked Python path that takes what it declines: the same results
bit for bit, and the same exception, type and text, for arguments that are refused."""
import pytest
import torch

from tests.helpers import decode_case, meta, rand_t

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ENTRIES = ("context_attention", "prefill_partial", "token_decode_attention", "decode_stage1", "decode_stage2", "kv_scatter",
           "register_decode_tokens", "register_tokens", "rms_norm", "silu_and_mul_inplace", "rotary_emb", "rotary_kv_write")


def _both(lsa, monkeypatch, make):
    """(outcome, whether an entry took the call) of make() through the native pass, and its outcome with every entry declining.  make()
    builds its arguments anew, calls an operator and returns the tensors it wrote."""
    from loongserve_amd import _native
    took = []

    def outcome():
        try:
            r = make()
        except Exception as e:
            return type(e), str(e)
        return [t.clone() for t in r]

    with monkeypatch.context() as m:
        for name in ENTRIES:
            real = getattr(_native, name)
            m.setattr(_native, name, lambda *a, real=real: (r := real(*a), took.append(r is not None))[0])
        native = outcome()
    with monkeypatch.context() as m:
        for name in ENTRIES:
            m.setattr(_native, name, lambda *a: None)
        checked = outcome()
    return native, any(took), checked


def _prefill(lsa, D=128, dtype=torch.float16, lens=(150, 33), **change):
    T, Hq, Hkv = sum(lens), 8, 2
    a = dict(q=rand_t((T, Hq, D), 1, dtype).to(DEV), k=rand_t((T, Hkv, D), 2, dtype).to(DEV), v=rand_t((T, Hkv, D), 3, dtype).to(DEV),
             m=torch.full((T, Hq), -float("inf"), device=DEV), l=torch.zeros((T, Hq), device=DEV), meta=[t.to(DEV) for t in meta(list(lens))],
             peers=1, max_q=max(lens))
    a["o"] = torch.empty_like(a["q"])
    kw = {k: v for k, v in change.items() if k not in a}
    for k, f in change.items():
        if k in a:
            a[k] = f(a[k])
    return a, kw


def _in_place(lsa, **change):
    a, kw = _prefill(lsa, **change)
    lsa.context_attention_fwd(a["q"], a["k"], a["v"], a["o"], *a["meta"], *a["meta"], a["peers"], a["max_q"], a["m"], a["l"], **kw)
    return a["o"], a["m"], a["l"]


def _partial(lsa, **change):
    a, kw = _prefill(lsa, **change)
    return lsa.prefill_attention_step(a["q"], a["k"], a["v"], *a["meta"], *a["meta"], a["peers"], a["max_q"], **kw)


def _fused(lsa, **change):
    B, Hq, Hkv, D, lens = 3, 8, 2, 128, [700, 33, 1025]
    q, kv, table, req, n = [t.to(DEV) for t in decode_case(77, B, Hq, Hkv, D, lens, 3000)]
    a = dict(q=q, k=kv[:, :Hkv], v=kv[:, Hkv:], table=table, req=req, n=n, mo=torch.zeros((5, B, Hq, D), device=DEV),
             ml=torch.zeros((5, B, Hq), device=DEV), out=None, lse=None)
    for k, f in change.items():
        a[k] = f(a[k])
    return lsa.longserve_token_decode_attention_flash_decoding(a["q"], a["table"], a["req"], a["n"], a["mo"], a["ml"], B, max(lens), Hq, D,
                                                               a["k"], a["v"], 256, a["out"], a["lse"])


def _stages(lsa, block=256, **change):
    B, Hq, Hkv, D, lens = 3, 8, 2, 128, [700, 33, 1025]
    q, kv, table, req, n = [t.to(DEV) for t in decode_case(78, B, Hq, Hkv, D, lens, 3000)]
    a = dict(q=q, mo=torch.zeros((5, B, Hq, D), device=DEV), ml=torch.zeros((5, B, Hq), device=DEV), o=torch.zeros((B, Hq, D), device=DEV),
             l=torch.zeros((B, Hq), device=DEV), n=n)
    for k, f in change.items():
        a[k] = f(a[k])
    c = lsa.longserve_cuda_kernels
    c.flash_decoding_stage1(a["mo"], a["ml"], a["q"], kv[:, :Hkv], kv[:, Hkv:], table, req, a["n"], max(lens), block)
    c.flash_decoding_stage2(a["o"], a["l"], a["n"], a["mo"], a["ml"], block)
    return a["mo"], a["ml"], a["o"], a["l"]


def _scatter(lsa, index=lambda t: t, src=lambda t: t, pool=lambda t: t):
    s, p = src(rand_t((50, 4, 64), 4).to(DEV)), pool(torch.zeros((80, 4, 64), dtype=torch.float16, device=DEV))
    lsa.kv_scatter(s, index(torch.arange(79, 29, -1, device=DEV)), p)
    return (p,)


def _register(lsa, prefill, mem=lambda t: t, table=lambda t: t, n=lambda t: t):
    lens, tb = n(torch.tensor([9, 4, 7], dtype=torch.int32, device=DEV)), table(torch.zeros((5, 12), dtype=torch.int32, device=DEV))
    req, slots = torch.tensor([3, 0, 4], dtype=torch.int32, device=DEV), mem(torch.arange(100, 120 if prefill else 103, device=DEV).int())
    if prefill:
        lsa.init_req_to_token_indexes(tb, req, lens, slots, torch.tensor([0, 9, 13], dtype=torch.int32, device=DEV), 9)
    else:
        lsa.copy_kv_index_to_req(tb, req, lens, slots)
    return (tb,)


def _steps(lsa, op, x=lambda t: t, w=lambda t: t, k=lambda t: t):
    c = lsa.longserve_cuda_kernels
    if op == "norm":
        return (c.rms_norm(x(rand_t((37, 512), 5).to(DEV)), w(rand_t((512,), 6).to(DEV)), 1e-5),)
    if op == "silu":
        io = x(rand_t((37, 512), 7).to(DEV))
        c.silu_and_mul_inplace(io)
        return (io,)
    q, kv = x(rand_t((37, 8, 128), 8).to(DEV)), k(rand_t((37, 4, 128), 9).to(DEV))
    cos, sin = w(rand_t((37, 64), 10).to(DEV)), rand_t((37, 64), 11).to(DEV)
    if op == "rotary":
        c.rotary_emb(q, kv, cos, sin)
        return q, kv
    pool, table = torch.zeros((90, 4, 128), dtype=torch.float16, device=DEV), torch.zeros((40, 9), dtype=torch.int32, device=DEV)
    lsa.rotary_emb_write_kv(q, kv, cos, sin, torch.arange(80, 43, -1, device=DEV), pool, table, torch.arange(37, device=DEV).int(),
                            torch.full((37,), 3, device=DEV).int(), decode=True)
    return q, kv, pool, table


# (operator, changes, does the native pass take it)
TAKEN = [
    (_in_place, {}), (_in_place, dict(dtype=torch.bfloat16)), (_in_place, dict(D=64)), (_in_place, dict(lens=(1,), total_q_len=1)),
    (_partial, {}), (_partial, dict(dtype=torch.bfloat16)), (_partial, dict(kv_splits=3)), (_partial, dict(sm_scale=0.5, D=32)),
    (_fused, {}), (_stages, {}), (_stages, dict(block=300)),
    (_scatter, {}), (_scatter, dict(index=lambda t: t.int())), (_register, dict(prefill=True)), (_register, dict(prefill=False)),
    (_register, dict(prefill=False, mem=lambda t: t.long())),
    (_steps, dict(op="norm")), (_steps, dict(op="silu")), (_steps, dict(op="rotary")), (_steps, dict(op="write")),
]
DECLINED = [
    (_in_place, dict(o=lambda t: t.float())), (_in_place, dict(meta=lambda t: [x.long() for x in t])), (_in_place, dict(total_q_len=-1)),
    (_in_place, dict(k=lambda t: t[:, :, :64])), (_in_place, dict(m=lambda t: t.half())), (_in_place, dict(q=lambda t: t.transpose(1, 2))),
    (_in_place, dict(k=lambda t: t.cpu())),
    (_partial, dict(accumulate=True)), (_partial, dict(v=lambda t: t.bfloat16())), (_partial, dict(k=lambda t: t[:, [0, 1, 1]], v=lambda t: t[:, [0, 1, 1]])),
    (_fused, dict(q=lambda t: t.float())), (_fused, dict(table=lambda t: t.long())), (_fused, dict(mo=lambda t: t[:, :2])),
    (_fused, dict(req=lambda t: t[:2])), (_fused, dict(n=lambda t: t.cpu())), (_fused, dict(mo=lambda t: t.half())),
    (_stages, dict(q=lambda t: t.float())), (_stages, dict(ml=lambda t: t[:4])), (_stages, dict(block=0)), (_stages, dict(n=lambda t: t.long())),
    (_scatter, dict(index=lambda t: t.short())), (_scatter, dict(index=lambda t: t[:40])), (_scatter, dict(pool=lambda t: t.float())),
    (_scatter, dict(src=lambda t: t.transpose(1, 2))), (_scatter, dict(src=lambda t: t[:0], index=lambda t: t[:0])),
    (_register, dict(prefill=True, mem=lambda t: t.long())), (_register, dict(prefill=False, table=lambda t: t.long())),
    (_register, dict(prefill=False, mem=lambda t: t[:2])), (_register, dict(prefill=True, n=lambda t: t.long())),
    (_steps, dict(op="norm", x=lambda t: t.float())), (_steps, dict(op="norm", w=lambda t: t[:504])), (_steps, dict(op="silu", x=lambda t: t[:, :511])),
    (_steps, dict(op="rotary", w=lambda t: t[:, :32])), (_steps, dict(op="rotary", k=lambda t: t[:30])), (_steps, dict(op="write", x=lambda t: t.float())),
    (_steps, dict(op="write", k=lambda t: t[:, :3])),
]


@pytest.mark.parametrize("i", range(len(TAKEN)))
def test_native_pass_and_checked_path_agree(lsa, monkeypatch, i):
    op, change = TAKEN[i]
    native, took, checked = _both(lsa, monkeypatch, lambda: op(lsa, **change))
    assert took and isinstance(checked, list), checked
    assert all(torch.equal(a, b) for a, b in zip(native, checked)) and len(native) == len(checked)


@pytest.mark.parametrize("i", range(len(DECLINED)))
def test_what_the_native_pass_declines_goes_the_checked_way(lsa, monkeypatch, i):
    op, change = DECLINED[i]
    native, _, checked = _both(lsa, monkeypatch, lambda: op(lsa, **change))
    if isinstance(checked, list):
        assert isinstance(native, list) and all(torch.equal(a, b) for a, b in zip(native, checked))
    else:
        assert native == checked
