"""CPU-only checks of the drop-in boundary: the C-ABI library loads and exports every
symbol include/lsattn.h declares, and argument validation rejects bad input without
touching a GPU."""
import ctypes as C
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_symbols():
    text = open(os.path.join(ROOT, "include", "lsattn.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(lsattn_[a-z0-9_]+)\s*\(", text)))


def test_importing_the_package_first_leaves_one_hip_runtime_in_the_process():
    """PyTorch-ROCm ships its own libamdhip64; the library links the system's.  Whatever the program imports first, the
    process must end up with one runtime (two: the library's launches find no device in theirs)."""
    import subprocess
    import sys
    code = ("import loongserve_amd, torch\n"
            "print(sorted({l.split()[-1] for l in open('/proc/self/maps') if 'libamdhip64' in l}))")
    out = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stderr[-2000:]
    paths = eval(out.stdout.strip().splitlines()[-1])
    assert len(paths) == 1, paths


def test_ceiling_library_exports_every_declared_symbol():
    """libls_ceiling.so (bench.py's measurement aids) exports what include/ls_ceiling.h declares."""
    import ctypes
    import torch  # noqa: F401  (first, so that this process keeps to one HIP runtime: see the test above)
    text = open(os.path.join(ROOT, "include", "ls_ceiling.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    names = sorted(set(re.findall(r"\b(ls_ceiling_[a-z0-9_]+)\s*\(", text)))
    assert len(names) == 5, names
    lib = ctypes.CDLL(os.path.join(ROOT, "loongserve_amd", "libls_ceiling.so"))
    for n in names:
        assert getattr(lib, n) is not None


def test_library_exports_every_declared_symbol():
    from loongserve_amd import _lib
    lib = _lib.load()
    names = _declared_symbols()
    assert len(names) >= 9
    assert set(names) == set(_lib.EXPORTS), (names, sorted(_lib.EXPORTS))
    for n in names:
        assert getattr(lib, n) is not None
    # LSATTN_VERSION of include/lsattn.h: the argument blocks as _lib.py declares them
    header = open(os.path.join(ROOT, "include", "lsattn.h")).read()
    assert lib.lsattn_version() == _lib.LSATTN_VERSION == int(re.search(r"#define LSATTN_VERSION (\d+)", header).group(1))
    assert lib.lsattn_strerror(0) == b"ok"
    assert b"invalid" in lib.lsattn_strerror(-1)


def test_native_argument_pass_is_built_for_the_same_interface(monkeypatch):
    """_native.so holds the argument blocks too: one that was built against another header is refused, as such a library is."""
    from loongserve_amd import _lib, _native
    header = open(os.path.join(ROOT, "include", "lsattn.h")).read()
    assert _native.LSATTN_VERSION == int(re.search(r"#define LSATTN_VERSION (\d+)", header).group(1))
    assert "int32_t dest_index_is_i64;" in header and _native.LSATTN_VERSION >= 4  # (version 3 had a reserved word there)
    monkeypatch.setattr(_lib, "_lib", None)
    for other in (_native.LSATTN_VERSION - 1, None):
        monkeypatch.setattr(_native, "LSATTN_VERSION", other)
        with pytest.raises(ImportError, match="interface version"):
            _lib.load()


def test_struct_layout_matches_header():
    # compile a tiny C program against the header and compare sizeof / offsetof with ctypes
    import subprocess
    import tempfile
    from loongserve_amd import _lib
    src = r'''
#include <stdio.h>
#include <stddef.h>
#include "lsattn.h"
int main(void) {
  printf("%zu %zu %zu %zu %zu\n", sizeof(lsattn_prefill_args), sizeof(lsattn_merge_args),
         sizeof(lsattn_decode_stage1_args), sizeof(lsattn_decode_stage2_args), sizeof(lsattn_kv_copy_register_args));
  printf("%zu %zu\n", sizeof(lsattn_decode_migration_args), offsetof(lsattn_decode_migration_args, b_seq_len));
  printf("%zu %zu\n", sizeof(lsattn_rotary_kv_write_args), offsetof(lsattn_rotary_kv_write_args, register_mode));
  printf("%zu %zu\n", sizeof(lsattn_tuning), offsetof(lsattn_tuning, decode_listed));
  printf("%zu %zu %zu %zu\n", sizeof(lsattn_merge_cuts_args), offsetof(lsattn_merge_cuts_args, ml_stride_h), offsetof(lsattn_prefill_args, o_cut_rows),
         offsetof(lsattn_prefill_args, total_q_rows));
  printf("%zu %zu %zu %zu %zu %zu\n", offsetof(lsattn_prefill_args, sm_scale), offsetof(lsattn_prefill_args, ml_stride_h),
         offsetof(lsattn_decode_stage1_args, req_to_tokens), offsetof(lsattn_decode_stage2_args, block_seq),
         offsetof(lsattn_kv_copy_register_args, req_to_tokens), offsetof(lsattn_kv_copy_register_args, should_register));
  return 0;
}'''
    with tempfile.TemporaryDirectory() as d:
        c = os.path.join(d, "t.c")
        open(c, "w").write(src)
        exe = os.path.join(d, "t")
        subprocess.check_call(["gcc", "-std=c99", "-I", os.path.join(ROOT, "include"), c, "-o", exe])
        out = subprocess.check_output([exe]).decode().split()
    sizes = [int(x) for x in out[:5]]
    mig = [int(x) for x in out[5:7]]
    rot = [int(x) for x in out[7:9]]
    tun = [int(x) for x in out[9:11]]
    cuts = [int(x) for x in out[11:15]]
    offs = [int(x) for x in out[15:]]
    assert cuts == [C.sizeof(_lib.MergeCutsArgs), _lib.MergeCutsArgs.ml_stride_h.offset, _lib.PrefillArgs.o_cut_rows.offset,
                    _lib.PrefillArgs.total_q_rows.offset]
    assert tun == [C.sizeof(_lib.Tuning), _lib.Tuning.decode_listed.offset]
    assert rot == [C.sizeof(_lib.RotaryKvWriteArgs), _lib.RotaryKvWriteArgs.register_mode.offset]
    assert mig == [C.sizeof(_lib.DecodeMigrationArgs), _lib.DecodeMigrationArgs.b_seq_len.offset]
    assert sizes == [C.sizeof(_lib.PrefillArgs), C.sizeof(_lib.MergeArgs), C.sizeof(_lib.DecodeStage1Args),
                     C.sizeof(_lib.DecodeStage2Args), C.sizeof(_lib.KvCopyRegisterArgs)]
    assert offs == [_lib.PrefillArgs.sm_scale.offset, _lib.PrefillArgs.ml_stride_h.offset,
                    _lib.DecodeStage1Args.req_to_tokens.offset, _lib.DecodeStage2Args.block_seq.offset,
                    _lib.KvCopyRegisterArgs.req_to_tokens.offset, _lib.KvCopyRegisterArgs.should_register.offset]


def test_validation_rejects_bad_arguments_without_gpu():
    from loongserve_amd import _lib
    lib = _lib.load()
    a = _lib.PrefillArgs()  # all null
    assert lib.lsattn_prefill_step(C.byref(a), None) == -1
    assert lib.lsattn_prefill_step(None, None) == -1
    d1 = _lib.DecodeStage1Args()
    assert lib.lsattn_decode_stage1(C.byref(d1), None) == -1
    mg = _lib.DecodeMigrationArgs()
    assert lib.lsattn_decode_migration_send(C.byref(mg), None) == -1
    assert lib.lsattn_decode_migration_recv(None, None) == -1
    rw = _lib.RotaryKvWriteArgs()
    assert lib.lsattn_rotary_kv_write(C.byref(rw), None) == -1
    assert lib.lsattn_rotary_kv_write(None, None) == -1
    cr = _lib.KvCopyRegisterArgs()
    assert lib.lsattn_kv_copy_register(C.byref(cr), None) == -1
    assert lib.lsattn_kv_ranges(None, None, None, 1, 0, None, None, None, None) == -1
    d2 = _lib.DecodeStage2Args()
    assert lib.lsattn_decode_stage2(C.byref(d2), None) == -1
    m = _lib.MergeArgs()
    assert lib.lsattn_lse_merge(C.byref(m), None) == -1
    assert lib.lsattn_kv_scatter(None, 0, None, 0, None, 0, 0, None) == -1
    assert lib.lsattn_bf16_to_f16_rows(None, 8, None, 8, 1, 8, None) == -1
    assert lib.lsattn_bf16_to_f16_rows(0x1000, 8, 0x2000, 8, 1, 16, None) == -1   # stride shorter than the row
    # slot allocator: sizes of the workspaces are host arithmetic, argument checks come before any launch
    assert lib.lsattn_pool_search_workspace_bytes(0) == 0
    assert lib.lsattn_pool_search_workspace_bytes(4096) == 16 + 28 + 4          # one workgroup of slots, padded to 16
    assert lib.lsattn_pool_search_workspace_bytes(2_500_000) >= 16 + 611 * 28
    assert lib.lsattn_pool_refs_workspace_bytes(0) == 0
    assert lib.lsattn_pool_refs_workspace_bytes(257) == 2 * 16 + 1040
    assert lib.lsattn_pool_alloc(None, 8, 1, None, None, 0, None) == -1
    assert lib.lsattn_pool_alloc(0x1000, 8192, 1, 0x2000, 0x3000, 16, None) == -4  # workspace too small
    assert lib.lsattn_pool_find_contiguous(0x1000, 8192, 0, 0x2000, 0x3000, 1 << 20, None) == -1  # need >= 1
    assert lib.lsattn_pool_find_contiguous(0x1004, 8192, 1, 0x2000, 0x3000, 1 << 20, None) == -1  # misaligned state
    assert lib.lsattn_pool_update_refs(0x1000, 8, 0x2000, 4, 2, 0x3000, 0x4000, 1 << 20, None) == -1  # delta must be +-1
    assert lib.lsattn_pool_update_refs(0x1000, 8, 0x2000, 4, 1, 0x3000, 0x4000, 8, None) == -4
    assert b"workspace" in lib.lsattn_strerror(-4)
    # unsupported head_dim is reported as such (pointers are fake but never dereferenced)
    fake = 0x1000
    for f in ("q", "k", "v", "o", "lse", "q_b_start_loc", "q_b_seq_len", "q_first_token_global_idx", "kv_b_start_loc",
              "kv_b_seq_len", "kv_first_token_global_idx"):
        setattr(a, f, fake)
    a.batch, a.num_q_heads, a.num_kv_heads, a.head_dim, a.sp_peers, a.max_q_len = 1, 4, 2, 48, 1, 8
    a.o_dtype = _lib.LSATTN_F32
    assert lib.lsattn_prefill_step(C.byref(a), None) == -2
    # head sizes 16, 32 and 64 have a kernel of their own, which does not cut the KV chunk
    a.head_dim, a.kv_cuts, a.kv_cut_len, a.o_cut_rows = 64, 2, 64, 8
    assert lib.lsattn_prefill_step(C.byref(a), None) == -2
    a.kv_cuts = a.kv_cut_len = a.o_cut_rows = 0
    a.head_dim, a.num_kv_heads = 128, 3
    assert lib.lsattn_prefill_step(C.byref(a), None) == -1
    # K/V token strides must be positive and keep a 64-row tile within a 32-bit byte offset
    a.num_kv_heads = 2
    for f in ("q_stride_t", "q_stride_h", "k_stride_h", "v_stride_h", "o_stride_t", "o_stride_h"):
        setattr(a, f, 128)
    a.dtype = _lib.LSATTN_F16
    for ks, vs in ((0, 256), (256, -256), ((1 << 24) + 8, 256), (256, 1 << 25)):
        a.k_stride_t, a.v_stride_t = ks, vs
        assert lib.lsattn_prefill_step(C.byref(a), None) == -1, (ks, vs)
    # the chunk cut along the keys: fp32 partials only, whole 64-key tiles per cut, the cuts' rows apart
    a.k_stride_t = a.v_stride_t = 256
    a.kv_cuts, a.kv_cut_len, a.o_cut_rows = 4, 100, 8
    assert lib.lsattn_prefill_step(C.byref(a), None) == -1          # not a multiple of 64 keys
    a.kv_cut_len, a.o_cut_rows = 128, 0
    assert lib.lsattn_prefill_step(C.byref(a), None) == -1          # no room between the cuts' outputs
    a.o_cut_rows, a.kv_cuts = 8, 65
    assert lib.lsattn_prefill_step(C.byref(a), None) == -1          # more cuts than LSATTN_MAX_KV_CUTS
    a.kv_cuts = 4
    assert lib.lsattn_prefill_step_accumulate(C.byref(a), None) == -1  # the folding steps take no cuts
    mc = _lib.MergeCutsArgs()
    assert lib.lsattn_prefill_merge_cuts(C.byref(mc), None) == -1
    assert lib.lsattn_prefill_merge_cuts(None, None) == -1
    for f in ("o_parts", "lse_parts", "q_b_start_loc", "q_b_seq_len", "o", "lse"):
        setattr(mc, f, fake)
    mc.n_parts, mc.batch, mc.num_q_heads, mc.head_dim, mc.max_q_len, mc.part_rows = 2, 1, 4, 64, 8, 8
    mc.o_stride_t, mc.o_stride_h, mc.o_dtype = 512, 128, _lib.LSATTN_F32
    assert lib.lsattn_prefill_merge_cuts(C.byref(mc), None) == -2   # head_dim
    mc.head_dim, mc.mode = 128, 1
    assert lib.lsattn_prefill_merge_cuts(C.byref(mc), None) == -1   # mode 1 needs m, l and a 16-bit o
    mc.mode, mc.n_parts = 0, 65
    assert lib.lsattn_prefill_merge_cuts(C.byref(mc), None) == -1
    # the fused decode call refuses argument blocks that do not describe the same partials
    s1, s2 = _lib.DecodeStage1Args(), _lib.DecodeStage2Args()
    assert lib.lsattn_decode_attention(None, C.byref(s2), None) == -1
    s1.mid_o, s2.mid_o = 0x1000, 0x2000
    assert lib.lsattn_decode_attention(C.byref(s1), C.byref(s2), None) == -1
    s2.mid_o = 0x1000
    s1.seq_block_size, s2.block_seq = 256, 128
    assert lib.lsattn_decode_attention(C.byref(s1), C.byref(s2), None) == -1
    # stage 1 merges at most 16 blocks into one partial
    s3 = _lib.DecodeStage1Args()
    for f in ("mid_o", "mid_o_logexpsum", "q", "k", "v", "req_to_tokens", "b_req_idx", "b_seqlen"):
        setattr(s3, f, 0x1000)
    s3.batch, s3.num_q_heads, s3.num_kv_heads, s3.num_blocks, s3.head_dim = 1, 4, 2, 4, 128
    s3.max_seq_len, s3.seq_block_size, s3.max_len_in_batch, s3.dtype = 1024, 256, 1024, _lib.LSATTN_F16
    s3.k_stride_0 = s3.v_stride_0 = 512
    s3.k_stride_1 = s3.v_stride_1 = 128
    for bad in (-1, 17):
        s3.merge_blocks = bad
        assert lib.lsattn_decode_stage1(C.byref(s3), None) == -1, bad


def test_tuning_block_is_validated_and_named_values_match_the_header():
    """lsattn_set_tuning takes the values include/lsattn.h names, refuses others, and NULL restores the library's choices;
    the names the Python side uses stand for the header's numbers."""
    from loongserve_amd import _lib
    lib = _lib.load()
    header = open(os.path.join(ROOT, "include", "lsattn.h")).read()
    num = {k: int(v) for k, v in re.findall(r"#define (LSATTN_(?:PREFILL|DECODE)_[A-Z0-9_]+) (\d+)", header)}
    want = {("prefill_rows", "128"): "LSATTN_PREFILL_ROWS_128", ("prefill_rows", "256"): "LSATTN_PREFILL_ROWS_256",
            ("prefill_rows", "half"): "LSATTN_PREFILL_ROWS_HALF", ("prefill_order", "tile"): "LSATTN_PREFILL_ORDER_TILE",
            ("prefill_order", "head"): "LSATTN_PREFILL_ORDER_HEAD", ("prefill_pack", "off"): "LSATTN_PREFILL_PACK_OFF",
            ("decode_stage1", "lane"): "LSATTN_DECODE_STAGE1_LANE", ("decode_stage1", "mfma"): "LSATTN_DECODE_STAGE1_MFMA",
            ("decode_stage1", "split"): "LSATTN_DECODE_STAGE1_SPLIT", ("decode_listed", "off"): "LSATTN_DECODE_LISTED_OFF",
            ("decode_listed", "on"): "LSATTN_DECODE_LISTED_ON", ("decode_listed", "shares"): "LSATTN_DECODE_LISTED_SHARES"}
    assert len(num) == len(want)
    for (field, name), macro in want.items():
        assert _lib.TUNING_VALUES[field][name] == num[macro]
        assert _lib.TUNING_VALUES[field][None] == 0
    try:
        t = _lib.Tuning()
        for field, top in (("prefill_rows", 3), ("prefill_order", 2), ("prefill_pack", 1), ("decode_stage1", 3), ("decode_listed", 3)):
            for bad in (-1, top + 1):
                t = _lib.Tuning()
                setattr(t, field, bad)
                assert lib.lsattn_set_tuning(C.byref(t)) == -1, (field, bad)
            t = _lib.Tuning()
            setattr(t, field, top)
            assert lib.lsattn_set_tuning(C.byref(t)) == 0
        t = _lib.Tuning()
        t.reserved[1] = 1
        assert lib.lsattn_set_tuning(C.byref(t)) == -1
        with pytest.raises(ValueError):
            _lib.set_tuning(prefill_rows="512")
        with pytest.raises(ValueError):
            _lib.set_tuning(no_such_choice="x")
    finally:
        assert lib.lsattn_set_tuning(None) == 0


def test_library_reads_no_environment_variable():
    """The launch choices come from lsattn_set_tuning alone: no source of the library calls getenv."""
    csrc = os.path.join(ROOT, "loongserve_amd", "csrc")
    for name in os.listdir(csrc):
        if name.endswith((".hip", ".h")):
            assert "getenv" not in open(os.path.join(csrc, name)).read(), name


def test_python_wrappers_reject_cpu_tensors():
    import torch
    import loongserve_amd as lsa
    q = torch.zeros(4, 2, 128, dtype=torch.float16)
    i = torch.zeros(1, dtype=torch.int32)
    with pytest.raises(ValueError):
        lsa.prefill_attention_step(q, q, q, i, i, i, i, i, i, 1, 4, out=torch.zeros(4, 2, 128), lse=torch.zeros(4, 2))
    with pytest.raises(ValueError):
        lsa.longserve_cuda_kernels.flash_decoding_stage1(torch.zeros(1, 1, 2, 128), torch.zeros(1, 1, 2), q[:1], q, q,
                                                         torch.zeros(1, 4, dtype=torch.int32), i, i, 4, 4)


def test_fused_decode_split_rule():
    """The fused decode call may split the context more coarsely than BLOCK_SEQ, but only while the launch keeps enough
    workgroups; the stage functions called on their own never change the block size they are given."""
    from loongserve_amd.decoding import FUSED_LONG_SPLIT_TOKENS, _fused_block_seq
    assert _fused_block_seq(256, 64, 32768, 8) == 1024           # config 3: 64 x 32 blocks x 2 task groups
    assert _fused_block_seq(256, 1, 4096, 8) == 256              # a single short request: nothing to spare
    assert _fused_block_seq(256, 16, 8192, 8) == 1024            # 16 x 8 blocks x 2 task groups = one workgroup per CU
    assert _fused_block_seq(256, 1, 131072, 8) == 1024
    assert _fused_block_seq(256, 1, 32768, 8) == 256
    assert _fused_block_seq(256, 1, 1048576, 8) == 4096          # very long contexts: up to 4096 while >= 64 blocks remain
    assert _fused_block_seq(256, 4, 131072, 32) == 2048
    assert _fused_block_seq(256, 16, 32768, 8) == 1024
    assert _fused_block_seq(2048, 64, 32768, 8) == 2048          # never below what the caller asked for
    assert _fused_block_seq(256, 64, 524288, 8) == 4096          # up to 64 requests may go beyond 1024
    assert _fused_block_seq(256, 256, 131072, 8) == 1024         # larger batches stay there: the likelier to hold one long request among short ones
    assert _fused_block_seq(16, 4096, 16, 8) == 16
    for bs in (1, 16, 64, 256):
        got = _fused_block_seq(bs, 1 << 14, 1 << 20, 32)
        assert got % bs == 0 and got <= max(FUSED_LONG_SPLIT_TOKENS, bs)


def test_extension_module_resolves_by_its_reference_name():
    """`import longserve_cuda_kernels`, as loongserve/models/llama/triton_kernel/longserve_flash_decoding_stage1.py:4 does."""
    import importlib
    m = importlib.import_module("longserve_cuda_kernels")
    from loongserve_amd import longserve_cuda_kernels as real
    for name in ("flash_decoding_stage1", "flash_decoding_stage2", "rms_norm", "silu_and_mul_inplace", "rotary_emb", "ffn_block",
                 "hello_world"):
        assert getattr(m, name) is getattr(real, name)


def test_kv_split_count_from_shapes():
    """The split of a short-query step along the keys is chosen from shapes alone (no device read-back)."""
    from loongserve_amd.ops import kv_split_count
    assert kv_split_count(1, 32, 16384, 16384) == 1          # config 2: 4096 workgroups
    assert kv_split_count(1, 32, 2048, 2048) == 1            # config 1: enough workgroups, few keys
    assert kv_split_count(1, 32, 100, 131072) == 8           # one 100-row chunk against 131072 keys: 32 workgroups -> one round of 256
    assert kv_split_count(1, 32, 100, 131072, 8) == 8        # GQA 32/8: four heads side by side, 8 x 4 workgroups of 32 positions
    assert kv_split_count(1, 32, 16, 131072, 8) == 32        # 16 rows: 8 workgroups; cuts of at least 4096 keys
    assert kv_split_count(1, 32, 16, 20000, 8) == 4
    assert kv_split_count(1, 8, 100, 20000) == 4             # cuts of at least 4096 keys
    assert kv_split_count(4, 32, 128, 100000) == 2           # 128 workgroups: two cuts
    assert kv_split_count(1, 100, 128, 100000) == 5          # 100 workgroups: two rounds of five cuts walk less than one round of two
    assert kv_split_count(1, 32, 100, 4096) == 1             # short KV
    assert kv_split_count(0, 32, 100, 100000) == 1


def test_cuts_are_bounded_by_the_memory_for_their_parts():
    """What the operators choose by themselves: never more parts than the caller's workspace holds, kv_split_count where it is a
    pair of tensors or holds fewer than that (the operators cap or refuse it then), one for short chunks."""
    torch = pytest.importorskip("torch")
    from loongserve_amd.ops import _choose_cuts, kv_split_count
    q = torch.empty((64, 8, 128), dtype=torch.float16, device="meta")
    for rows in (8192, 20000, 100000):
        k = torch.empty((rows, 1, 128), dtype=torch.float16, device="meta")
        sized = kv_split_count(1, 8, 64, rows, 1)
        free = _choose_cuts(q, k, 1, 64, None, None)
        assert 1 < sized <= free <= 64 and rows // free >= 512
        for held in (1, sized - 1, sized, sized + 1, 64):
            got = _choose_cuts(q, k, 1, 64, None, torch.empty(held * 64 * 8 * 129, device="meta"))
            assert got == sized if held < sized else got <= held
        assert _choose_cuts(q, k, 1, 64, None, (None, None)) == sized
        assert _choose_cuts(q, k, 1, 64, 8191, None) == 1
        assert _choose_cuts(q, k, 0, 64, None, None) == 1
    assert _choose_cuts(torch.empty((4096, 32, 128), device="meta"), k, 8, 4096, None, None) == 1


def test_operators_cut_no_launch_that_kv_split_count_leaves_whole():
    """A launch that is not cut takes no memory for parts; the ones that are take no more, over these shapes, than kv_split_count's
    counts may take."""
    torch = pytest.importorskip("torch")
    from loongserve_amd.ops import _choose_cuts, kv_split_count
    most, most_sized, whole = 0, 0, 0
    for batch in (1, 2, 3, 4, 8):
        for rows in (1, 64, 200, 500, 896, 1024, 1100, 1792, 2047):
            for keys in (8191, 8192, 9000, 20000, 100000):
                for Hq, Hkv in ((32, 32), (32, 8), (64, 8), (8, 1)):
                    q = torch.empty((batch * rows, Hq, 128), dtype=torch.float16, device="meta")
                    k = torch.empty((keys, Hkv, 128), dtype=torch.float16, device="meta")
                    for held in (None, torch.empty(64 * q.numel() * 2, device="meta")):
                        for given in (None, keys):
                            got = _choose_cuts(q, k, batch, rows, given, held)
                            sized, part = kv_split_count(batch, Hq, rows, keys, Hkv), batch * rows * Hq * 129 * 4
                            if sized == 1:
                                assert got == 1, (batch, rows, keys, Hq, Hkv)
                                whole += 1
                            else:
                                most, most_sized = max(most, got * part), max(most_sized, sized * part)
    assert whole and 0 < most <= most_sized < 256 << 20, (most, most_sized)


def test_cut_count_of_a_step():
    """The library's count: within what the memory holds, a cut no shorter than 512 keys, one where the arguments describe no step; the
    counts that were measured at some lengths."""
    from loongserve_amd import _lib
    count = _lib.load().lsattn_prefill_cut_count
    assert count(1, 32, 8, 64, 8192, 64) == 10 and count(1, 32, 8, 500, 65000, 64) == 4 and count(1, 32, 8, 500, 65000, 2) == 2
    assert count(1, 8, 1, 64, 17467, 64) in range(16, 25) and count(1, 8, 1, 209, 26261, 64) == 16
    for args in ((0, 32, 8, 64, 8192, 64), (1, 32, 0, 64, 8192, 64), (1, 32, 5, 64, 8192, 64), (1, 32, 8, 0, 8192, 64), (1, 32, 8, 64, 0, 64),
                 (1, 32, 8, 64, 8192, 0), (1, 32, 8, 64, 8192, -3), (1, 32, 8, 64, 1023, 64)):
        assert count(*args) == 1, args
    for rows in (1, 64, 500, 2047):
        for keys in (1024, 8192, 100000, 2 ** 31 - 1):
            for most in (1, 3, 64, 1000):
                assert 1 <= count(1, 8, 1, rows, keys, most) <= min(most, keys // 512, 64)


def _route(batch, max_q, heads, head_dim=128, total_q=0, total_kv=0, max_kv=0, dtype=0, v_is_f16=0, cuts=0, m=None):
    from loongserve_amd import _lib
    a = _lib.PrefillArgs()
    a.batch, a.max_q_len, a.head_dim, a.dtype, a.v_is_f16, a.kv_cuts = batch, max_q, head_dim, dtype, v_is_f16, cuts
    a.num_q_heads, a.num_kv_heads = heads
    a.total_q_rows, a.total_kv_rows, a.max_kv_len, a.m = total_q, total_kv, max_kv, m
    return _lib.load().lsattn_prefill_route(C.byref(a))


SMALL_16, SMALL_32, SMALL_TURNS, ROWS_256, ROWS_128, HALF, HALF_FOLDED = range(1, 8)


def test_short_prompts_kernel_goes_by_the_longest_request():
    """The kernel of short prompts runs where no request can have more than 1024 keys: what the K buffer holds beyond the query rows may
    all belong to one request, unless the caller bounds the lengths (16 requests of 64 rows, one behind 15000 keys: 145 -> 264 us in it)."""
    heads = (32, 8)
    assert _route(1, 100, (32, 32), total_q=100, total_kv=100) == SMALL_16
    assert _route(16, 64, heads, total_q=1024, total_kv=1024) == SMALL_16
    assert _route(16, 64, heads, total_q=1024, total_kv=15960) == ROWS_128
    assert _route(8, 64, heads, total_q=512, total_kv=448 + 7500) == ROWS_128
    assert _route(2, 100, heads, total_q=200, total_kv=2000) == ROWS_128  # (one of them behind 1900)
    assert _route(2, 100, heads, total_q=4096, total_kv=2000) == ROWS_128  # (a loose bound of the rows proves nothing)
    assert _route(8, 64, heads, total_q=512, total_kv=4800) == ROWS_128
    assert _route(8, 64, heads, total_q=512, total_kv=4800, max_kv=600) == SMALL_16
    assert _route(8, 64, heads, total_q=512, max_kv=1024) == SMALL_16
    assert _route(8, 64, heads, total_q=512, max_kv=1025) == ROWS_128
    assert _route(8, 64, heads, total_kv=1024) == SMALL_16 and _route(8, 64, heads, total_kv=1025) == ROWS_128
    assert _route(8, 64, heads) == _route(8, 64, heads, total_q=512) == ROWS_128  # (nothing known of the keys)
    assert _route(1, 768, heads, total_q=768, total_kv=1024) == SMALL_16 and _route(1, 768, heads, total_q=768, total_kv=1025) == ROWS_128
    assert _route(1, 769, heads, total_q=769, total_kv=769) == ROWS_128


def test_short_prompts_kernel_goes_by_the_workgroups_and_the_longest_prompt():
    """With 32 positions per wave it takes prompts of up to 768 tokens that are too many for 16, up to 1024 from three workgroups per CU
    on, up to 1280 from four to ten; ragged batches from a half, then a whole one more."""
    small = (SMALL_16, SMALL_32, SMALL_TURNS)
    heads = (32, 8)  # (32 positions of four heads: 8 workgroups per 32 tokens)
    own = lambda batch, n, heads=heads, **kw: _route(batch, n, heads, total_q=batch * n, total_kv=batch * n, **kw)
    mixed = lambda batch, n, total, heads=heads: _route(batch, n, heads, total_q=total, total_kv=total)
    assert own(2, 640) == own(2, 704) == own(2, 768) == SMALL_16 and own(3, 640) == own(3, 704) == own(4, 768) == SMALL_32  # 640, 704, 768 | 960 ..
    assert mixed(4, 700, 1216) == SMALL_16 and mixed(4, 700, 1217) == SMALL_TURNS                          # 640 and 648, of which some are short
    assert own(2, 768, (40, 40)) == SMALL_16 and own(3, 768, (32, 32)) == SMALL_32                       # 960 and 1152
    assert mixed(4, 768, 2000, (32, 32)) == SMALL_16                                                     # 1152
    assert own(3, 992) not in small and own(3, 1024) == SMALL_32                                         # 744 and 768 of 32
    assert mixed(8, 1024, 3296) not in small and mixed(8, 1024, 3297) in small                           # 888 and 896
    assert own(4, 1025) == SMALL_32 and own(3, 1025) not in small                                        # 1056 and 792
    assert own(8, 1280) == SMALL_32 and own(9, 1280) not in small and own(8, 1281) not in small          # 2560 and 2880
    assert mixed(12, 1280, 4736) not in small and mixed(12, 1280, 4737) in small and mixed(16, 1280, 16000) in small  # 1280, 1288 and 4128
    assert _route(8, 2049, heads, total_q=5000, total_kv=5000) == ROWS_256
    assert _route(16, 1000, heads, total_q=16000, total_kv=17100) == HALF  # (one of them behind 1100 more)
    assert _route(16, 1000, heads, total_q=16000) == _route(16, 1000, heads) == HALF  # (nothing known of the keys)
    assert _route(70000, 16, heads, total_q=70000 * 16, total_kv=70000 * 16) not in small  # (past the grid's index)


def test_prompts_that_lasted_longer_in_the_short_kernel_are_left_to_the_other():
    """Launches that took 2 to 31 % longer in it than in the 128-wide kernel (microseconds, that kernel | this one): 2 x 1594 32/8 partial 49.0 | 59.1, 19 x 1244 64/8 594 | 621, 2 x 1793 at most 47.9 | 62.5, and, as full steps of a ring, 5 x 1000 at most 32/8 up to twice as long
    with 16 positions per wave; and ragged batches that took longer with 32 positions than with 16 (15 x 356 at most 24/8 16.2 | 19.4)."""
    small = (SMALL_16, SMALL_32, SMALL_TURNS)
    for batch, n, heads in ((2, 1594, (32, 8)), (19, 1244, (64, 8)), (5, 1700, (32, 8)), (16, 2000, (32, 8))):
        for dtype in (0, 1):
            for m in (None, 256):
                assert _route(batch, n, heads, total_q=batch * n, total_kv=batch * n, dtype=dtype, m=m) not in small, (batch, n, heads)
    assert _route(2, 1793, (32, 8), total_q=3029, total_kv=3029) not in small and _route(16, 2000, (32, 8), total_q=14000, total_kv=14000) not in small
    assert _route(5, 1000, (32, 8), total_q=1400, total_kv=1400, m=256) not in small                     # 3 per CU of 16, one long prompt
    assert _route(15, 356, (24, 8), total_q=1785, total_kv=1785, dtype=1) == SMALL_16


def test_one_prompt_in_a_few_four_wave_workgroups_more_than_two_per_cu():
    one = lambda n, heads, **kw: _route(1, n, heads, total_q=n, **{"total_kv": n, **kw})
    assert [one(n, (32, 32)) for n in (2049, 2816, 2817, 4097)] == [HALF, HALF, ROWS_256, ROWS_256]
    assert [one(n, (32, 8)) for n in (2049, 2304, 2305, 4097)] == [HALF, HALF, ROWS_256, ROWS_256]
    assert one(6144, (11, 11)) == HALF and one(6145, (11, 11)) == ROWS_256
    assert one(2561, (32, 32), total_kv=2562) == one(2561, (32, 32), total_kv=0) == one(2561, (32, 32), cuts=2) == ROWS_256
    assert _route(2, 1100, (32, 32), total_q=2200, total_kv=2200) != HALF


def test_longer_prompts_in_few_workgroups_of_16_positions():
    """Beyond 768 tokens where 128-row workgroups would fill half the chip, or start a second round of few."""
    small = (SMALL_16, SMALL_32, SMALL_TURNS)
    one = lambda n, heads, dtype=0, **kw: _route(1, n, heads, total_q=n, total_kv=kw.pop("total_kv", n), dtype=dtype, **kw)
    assert one(769, (8, 1)) == one(1280, (8, 1)) == SMALL_16 and one(1281, (8, 1)) not in small          # one workgroup per CU and less
    assert one(1024, (8, 1), 1) == SMALL_16 and one(1025, (8, 1), 1) not in small
    assert one(1024, (16, 16)) == SMALL_16 and one(1025, (16, 16)) not in small                          # 256 and 272 workgroups
    place = dict(m=256)  # (an in-place step has one; no pointer is followed)
    assert one(1000, (40, 40)) == one(1024, (40, 40), 1) == SMALL_16                                     # 640 workgroups, any epilogue
    assert one(1024, (32, 32), **place) not in small and one(1025, (32, 32), **place) == SMALL_16        # 512 and 544
    assert one(1025, (32, 32)) not in small and one(1025, (32, 32), 1) == SMALL_16
    assert one(1280, (32, 8), **place) == SMALL_16 and one(1281, (32, 8), **place) not in small          # 640 and 648
    assert one(1280, (32, 32), 1) == SMALL_16 and one(1281, (32, 32), 1, **place) not in small
    assert _route(2, 1000, (20, 20), total_q=1900, total_kv=1900) == _route(3, 1000, (20, 20), total_q=1900, total_kv=1900) == SMALL_16
    assert _route(3, 1000, (32, 8), total_q=1200, total_kv=1200) not in small                            # 624, ragged, four heads side by side
    assert one(1040, (32, 8), 1, **place) not in small
    assert _route(1, 1120, (32, 32), total_q=1120, total_kv=1280, **place) == SMALL_16                   # (keys beyond the rows)
    assert _route(1, 1120, (32, 32), total_q=1120, total_kv=1281, **place) not in small
    assert _route(1, 1120, (32, 32), total_q=1120, **place) not in small


def test_spare_rows_of_the_k_buffer_leave_the_order_of_the_grid_alone():
    """64-wide heads, ragged requests that take turns (ids of a tile a multiple of 32, which those of a bunch of one request are not): against a K
    buffer of many more rows than the requests have as against their own, with the bound on the rows and with one on the keys; behind
    contexts that the caller bounds, the K/V read counts."""
    for spare in (0, 1 << 17, 1 << 20):
        assert _route(8, 2000, (32, 8), 64, total_q=9000, total_kv=9000 + spare) == SMALL_TURNS
        assert _route(8, 2000, (32, 8), 64, total_q=9000, total_kv=9000 + spare, max_kv=2000) == SMALL_TURNS
    # (184 MB read, bunches of one request; 41 MB)
    assert _route(8, 20000, (32, 8), 64, total_q=90000, total_kv=1 << 20, max_kv=20000) == SMALL_32
    assert _route(8, 8000, (32, 8), 64, total_q=20000, total_kv=1 << 20, max_kv=8000) == SMALL_TURNS


def test_bunches_by_the_kv_that_is_read_have_two_rounds_of_workgroups():
    """64-wide heads, ragged, 16/16 heads, K/V of 73 MB: two bunches would be about a round of workgroups each, of which one ends with the longest
    request's alone (11 requests of at most 5345 tokens 193 us, whole 146); 266 MB on 32/8 are eight bunches of four rounds."""
    assert _route(6, 5345, (16, 16), 64, total_q=18652, total_kv=18652) == SMALL_TURNS    # (6 x 16 ids a tile are a multiple of 32, 3 x 16 are not)
    assert _route(8, 30000, (32, 8), 64, total_q=130000, total_kv=130000) == SMALL_32     # (8 x 8 are, 8 are not)


def test_prefill_route_names_a_kernel_for_every_step_and_none_for_others():
    assert _route(24, 256, (32, 32), total_q=1800, total_kv=1800) == SMALL_32
    assert _route(8, 3000, (32, 8), 64, total_q=16000, total_kv=16000) == SMALL_TURNS
    assert _route(8, 3000, (32, 8), 64, total_q=24000) == _route(8, 3000, (32, 8), 64) == SMALL_32
    assert _route(1, 100, (32, 32), 16) == SMALL_16
    assert _route(1, 2048, (32, 32)) == HALF_FOLDED and _route(16, 1024, (32, 8)) == HALF
    assert _route(1, 16384, (32, 32)) == ROWS_256 and _route(1, 500, (32, 8), cuts=2) == ROWS_128 and _route(1, 500, (32, 8), cuts=3) == ROWS_256
    assert _route(1, 100, (32, 8), dtype=1) == ROWS_256 and _route(1, 100, (32, 8), dtype=1, v_is_f16=1) == ROWS_128
    assert _route(0, 100, (32, 8)) == _route(1, 0, (32, 8)) == _route(1, 100, (32, 0)) == _route(1, 100, (32, 5)) == _route(1, 100, (32, 8), 80) == 0


def test_lone_prompts_past_1280_rows_fold_in_the_short_prompts_kernel():
    """One f16 prompt of up to 1472 rows in the in-place epilogue with a head per workgroup, in the third workgroup of 64 rows per CU; up to one per
    CU, where two waves share a tile, any request of 512 to 2304 keys (bf16 2048).  Nothing else past 1280, or beside another request."""
    lone = lambda n, heads, kv=None, **kw: _route(1, n, heads, total_q=n, total_kv=kv or n, **kw)
    bf16 = dict(dtype=1, v_is_f16=1, m=256)
    for n in (1281, 1410, 1472):
        assert lone(n, (32, 32), m=256) == SMALL_16 and lone(n, (32, 32)) == lone(n, (8, 1)) == ROWS_128
        assert lone(n, (32, 32), **bf16) == lone(n, (32, 8), m=256) == ROWS_128
        assert lone(n, (32, 32), kv=n + 1, m=256) == lone(n, (32, 32), kv=1000, m=256) == ROWS_128
        assert _route(2, n, (32, 32), total_q=2 * n, total_kv=2 * n, m=256) not in (SMALL_16, SMALL_32)
    assert lone(1473, (32, 32), m=256) == lone(1300, (20, 20), m=256) == ROWS_128  # (1.6 workgroups of 64 rows per CU)
    assert lone(2048, (8, 1), m=256) == lone(2304, (4, 1), m=256) == SMALL_16 and lone(2049, (8, 1), m=256) == lone(2305, (4, 1), m=256) == ROWS_128
    assert lone(1025, (8, 1), **bf16) == lone(2048, (8, 1), **bf16) == SMALL_16 and lone(2049, (4, 1), **bf16) == lone(1025, (8, 1), dtype=1, v_is_f16=1) == ROWS_128
    assert lone(200, (32, 8), kv=1224, m=256) == lone(200, (32, 8), kv=2304, m=256) == SMALL_16
    assert lone(200, (32, 8), kv=2305, m=256) == lone(200, (32, 8), kv=1224) == _route(2, 100, (32, 8), total_q=200, total_kv=1224, m=256) == ROWS_128


def test_lone_prompts_of_a_few_workgroups_past_two_per_cu():
    """Folded in place, where 256-row workgroups end in a round of a few: two of four waves per CU, or three rounds of the split shape past 6144 rows."""
    lone = lambda n, heads, m=256: _route(1, n, heads, total_q=n, total_kv=n, m=m)
    assert lone(2500, (32, 8)) == lone(2816, (32, 8)) == HALF and lone(2817, (32, 8)) == lone(2500, (32, 8), None) == ROWS_256  # (704 workgroups of 128 rows)
    assert lone(2944, (32, 32)) == HALF and lone(2945, (32, 32)) == lone(2944, (32, 32), None) == ROWS_256                      # (736)
    assert lone(1400, (64, 8)) == ROWS_256 and lone(5000, (16, 2)) == HALF  # (several heads, up to 1536 rows: up to 576)
    assert lone(6144, (14, 14)) == HALF and lone(6145, (14, 14)) == ROWS_256 and lone(6272, (13, 13)) == ROWS_128
    assert lone(8300, (8, 1)) == lone(10752, (8, 1)) == ROWS_128 and lone(10753, (8, 1)) == lone(8300, (8, 1), None) == ROWS_256  # (672)
    assert lone(1290, (40, 40)) == lone(1408, (36, 36)) == lone(1300, (40, 40), None) == HALF and lone(1409, (36, 36)) == ROWS_128
    assert _route(1, 2500, (32, 8), total_q=2500, total_kv=2600, m=256) == ROWS_256 and _route(2, 1250, (32, 8), total_q=2500, total_kv=2500, m=256) != HALF


def test_lone_prompts_of_heads_side_by_side_keep_256_rows():
    """Between three halves and seven quarters of a 128-row workgroup per CU the four-wave shape takes one head per workgroup only."""
    lone = lambda n, heads, m=256: _route(1, n, heads, total_q=n, total_kv=n, m=m)
    assert lone(800, (64, 8)) == lone(800, (64, 8), None) == lone(863, (64, 8)) == ROWS_256
    assert lone(1100, (44, 44)) == HALF


def test_equal_prompts_fill_a_third_workgroup_per_cu():
    """Equal f16 requests in place: 769 to 1024 rows from two workgroups of 32 positions per CU on, up to 1280 from 2.6 on, up to three."""
    step = lambda b, n, heads, m=256, total=None, **kw: _route(b, n, heads, total_q=total or b * n, total_kv=total or b * n, m=m, **kw)
    assert step(9, 1024, (8, 8)) == step(10, 769, (8, 8)) == SMALL_32 and step(8, 1024, (8, 8)) == ROWS_256  # (576, 560, 512)
    assert step(9, 1280, (8, 8)) == SMALL_32 and step(8, 1280, (8, 8)) == ROWS_256  # (720, 640)
    assert step(10, 1280, (8, 8)) != SMALL_32 and step(9, 1281, (8, 8)) != SMALL_32  # (800)
    assert step(9, 1024, (8, 8), m=None) == step(9, 1024, (8, 8), dtype=1) == ROWS_256
    assert step(9, 1024, (8, 8), total=8294) != SMALL_32  # (nine tenths of 9216)


def test_ragged_batches_folded_in_place_by_four_waves():
    """Ragged requests of up to 2048 rows against as many keys, from a workgroup of 128 rows per CU on (three halves where it would be the split shape's)."""
    step = lambda n, total, heads=(32, 8), m=256, **kw: _route(4, n, heads, total_q=total, total_kv=kw.pop("total_kv", total), m=m, **kw)
    assert step(2048, 5000) == HALF and step(2049, 5000) == step(2048, 5000, m=None) == step(2048, 5000, total_kv=5001) == ROWS_256
    assert step(2048, 7372) == HALF and step(2048, 7373) == ROWS_256  # (nine tenths of 8192)
    assert step(1900, 2000, (8, 1)) == ROWS_128  # (1.0 per CU)


def test_ragged_batches_of_few_workgroups_keep_their_shape():
    """Folded in place by four waves from nine halves of a workgroup of 128 rows per CU on, of eight requests from three and of sixteen from one on; not in place of the split shape."""
    step = lambda b, n, total, heads, m=256: _route(b, n, heads, total_q=total, total_kv=total, m=m)
    assert step(4, 1973, 3262, (14, 2)) == step(5, 1704, 2399, (16, 16)) == ROWS_128        # (1.6 and 1.5 per CU, the split shape's)
    assert step(2, 1523, 1713, (32, 32)) == step(3, 975, 1200, (32, 8)) == ROWS_256         # (1.8 and 1.3)
    assert step(4, 2048, 4448, (32, 8)) == ROWS_256 and step(4, 2048, 4449, (32, 8)) == HALF  # (143 and 144 tiles of 32 rows)
    assert step(8, 1500, 2784, (32, 8)) == ROWS_256 and step(8, 1500, 2785, (32, 8)) == HALF  # (95 and 96)
    assert step(15, 1200, 2700, (32, 8)) == HALF and step(16, 900, 4000, (8, 1)) == step(20, 840, 5000, (8, 1)) == HALF  # (1.1 and 1.4)
    assert step(15, 1200, 2400, (32, 8)) == ROWS_256                                        # (2.8)
    assert step(3, 1959, 3000, (64, 8)) == step(2, 1959, 2565, (64, 8)) == ROWS_256         # (two and three requests: full steps 139 -> 147 us)


def test_equal_prompts_barely_past_two_workgroups_per_cu_keep_256_rows():
    """Equal f16 requests in place fill a third workgroup of 32 positions per CU from 33/16 on."""
    step = lambda b, n, heads: _route(b, n, heads, total_q=b * n, total_kv=b * n, m=256)
    assert step(5, 832, (16, 1)) == ROWS_256 and step(5, 833, (16, 1)) == SMALL_32  # (26 and 27 tiles of 32 rows: 520 and 540 workgroups)
    assert step(11, 1024, (6, 6)) == SMALL_32                                     # (528)


def test_argument_blocks_in_the_documents_match_the_header():
    """Every ctypes mirror that a document at the top of the tree shows has the fields, in order and type, of the block this package passes, its example names a value for each
    of them, and the interface version beside it is the header's."""
    import glob
    from loongserve_amd import _lib
    found = 0
    for path in glob.glob(os.path.join(ROOT, "*.md")):
        text = open(path).read()
        for version in re.findall(r"lsattn_version\(\) == LSATTN_VERSION`? \((\d+)\)", text):
            assert int(version) == _lib.LSATTN_VERSION, path
        for name, body in re.findall(r"^class (\w+)\(C\.Structure\):.*?\n((?:    .*\n)+)", text, flags=re.M):
            space = {"C": C}
            exec("class %s(C.Structure):\n%s" % (name, body), space)
            assert space[name]._fields_ == getattr(_lib, name)._fields_, (path, name)
            calls = re.findall(r"= %s\((.*?)\)[ ]*(?:#.*)?\n(?=rc)" % name, text, flags=re.S)
            for call in calls:
                depth, args = 0, 1
                for ch in call:
                    depth += (ch in "([") - (ch in ")]")
                    args += ch == "," and depth == 0
                assert args == len(space[name]._fields_), (path, name, args)
                found += 1
    assert found >= 1


def test_lone_requests_of_few_rows_under_a_loose_bound_keep_their_shape():
    """One request goes to the short prompts' kernel past 1280 keys for the two waves that share its tiles, which are counted by the bound on its rows."""
    step = lambda n, total, kv: _route(1, n, (32, 8), total_q=total, total_kv=kv, m=256)
    assert step(200, 200, 2000) == step(512, 200, 2000) == SMALL_16 and step(1400, 200, 2000) == ROWS_128  # (at most 13, 32 and 88 workgroups per head)
    assert step(200, 200, 511) == SMALL_16
