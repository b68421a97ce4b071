"""CPU-only checks of the C-ABI boundary: the library loads, exports exactly what
include/pariskv_hip.h declares, and the Python binding has a prototype for each."""
import ctypes
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "pariskv_hip.h")


def declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(pkv_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_expected_surface():
    names = declared_functions()
    for must in ("pkv_encode_append", "pkv_query_prep_lut", "pkv_update_cache_cnt", "pkv_bucket_topk", "pkv_topk_f32",
                 "pkv_rerank4", "pkv_gather_uva", "pkv_gather_hbm", "pkv_gather_cpu", "pkv_retrieve"):
        assert must in names


def test_library_exports_every_declared_symbol():
    from pariskv_amd import _lib

    if not os.path.exists(_lib.SO_PATH):
        _lib.build()
    handle = ctypes.CDLL(_lib.SO_PATH)
    for name in declared_functions():
        assert hasattr(handle, name), f"{name} declared in the header but not exported"
        assert name in _lib.PROTOTYPES, f"{name} has no ctypes prototype"
    assert sorted(_lib.PROTOTYPES) == declared_functions()
    assert _lib.lib().pkv_version() >= 1


def test_every_declaration_cites_the_reference():
    text = open(HEADER).read()
    # each documented entry point names a reference file:line (or says it has no counterpart)
    blocks = re.findall(r"/\*(.*?)\*/\s*(?:size_t|int)\s+(pkv_[a-z0-9_]+)\s*\(", text, flags=re.S)
    assert len(blocks) >= 15
    for comment, name in blocks:
        assert re.search(r"\.(cu|py|cpp):\d+", comment) or "no counterpart" in comment.lower() or name in (
            "pkv_host_free", "pkv_host_device_pointer", "pkv_retrieve_ws_view"), name


def test_host_side_argument_errors_without_gpu():
    """Pure host validation paths return error codes and messages (no kernel is launched)."""
    from pariskv_amd import _lib

    L = _lib.lib()
    assert L.pkv_bucket_topk(None, 0, 1, 10, 5, None, None, 0, None) == _lib.EINVAL
    assert b"null pointer" in L.pkv_last_error()
    assert L.pkv_retrieve(None, None, 0, None) == _lib.EINVAL
    assert L.pkv_retrieve_ws_bytes(32, 131072, 4096, 1024) > 32 * 131072
    assert L.pkv_retrieve_ws_bytes(32, 100, 200, 10) == 0  # n_cand > n_keys
    with pytest.raises(RuntimeError, match="pariskv_hip error"):
        _lib.check(L.pkv_gather_cpu(None, None, None, None, None, 1, 1, 1, 1, 1, 2, 1))
    assert L.pkv_adaptive_decode_step(None, None, 0, None, None, None) == _lib.EINVAL
    a, ad, aa = _lib.RetrieveArgs(), _lib.AdaptiveArgs(), _lib.AttnArgs()
    a.out_ids = 8  # a final top-k was asked for: not the candidates-only form
    assert L.pkv_adaptive_decode_step(a, None, 0, ad, aa, None) == _lib.EINVAL
    assert b"candidates-only" in L.pkv_last_error()
    assert L.pkv_dense_logits(None, 1, 1, 1, 1, None, 0, 0, 1, 1.0, None, 1, None) == _lib.EINVAL
    assert L.pkv_adaptive_topk(None, 0, None, 0, 0, None, 0, 1.0, None, None, 0, 0, 0, None, 10, 0.9, 5, 1, None, None,
                               6, 5, None, 0, None, 0, None) == _lib.EINVAL
    assert b"clamp" in L.pkv_last_error()


def test_struct_mirrors_have_the_library_sizes():
    from pariskv_amd import _lib

    L = _lib.lib()
    for which, mirror in enumerate((_lib.AttnSegment, _lib.AttnArgs, _lib.RetrieveArgs, _lib.AdaptiveArgs)):
        assert L.pkv_struct_bytes(which) == ctypes.sizeof(mirror) > 0
    assert L.pkv_struct_bytes(4) == 0


def test_gather_cpu_host_function():
    """pkv_gather_cpu is host code: exercised fully on the CPU (gather_cpu.cpp contract)."""
    import torch

    from pariskv_amd.cache_hub.gather import load_gather_ext

    ext = load_gather_ext()
    g = torch.Generator().manual_seed(0)
    src = torch.randn(2, 3, 50, 128, generator=g).to(torch.bfloat16)
    idx = torch.randint(0, 50, (2, 3, 7), generator=g)
    out = torch.empty(2, 3, 7, 128, dtype=torch.bfloat16)
    ext.gather_kv_out_cpu(src, idx, out)
    assert torch.equal(out, torch.gather(src, 2, idx.unsqueeze(-1).expand(-1, -1, -1, 128)))
    src_t = torch.randn(2, 3, 128, 50, generator=g).transpose(2, 3)  # non-contiguous rows
    out32 = torch.empty(2, 3, 7, 128)
    ext.gather_kv_out_cpu(src_t, idx, out32)
    assert torch.equal(out32, torch.gather(src_t, 2, idx.unsqueeze(-1).expand(-1, -1, -1, 128)))
    idx[0, 0, 0] = 50
    with pytest.raises(RuntimeError, match="out of bounds"):
        ext.gather_kv_out_cpu(src, idx, out)


def test_gather_cpu_equals_the_reference_build():
    """pkv_gather_cpu and the oracle's gather_rows against the reference's own gather_cpu.cpp, compiled by
    oracle/build_ref.py into oracle/_ref (skipped where that build is absent)."""
    import numpy as np
    import torch

    from oracle import build_ref
    from oracle import pkv_oracle as O
    from pariskv_amd.cache_hub.gather import load_gather_ext

    ref = build_ref.load()
    if ref is None:
        pytest.skip("oracle/_ref is not built (python oracle/build_ref.py needs the reference tree)")
    ext = load_gather_ext()
    g = torch.Generator().manual_seed(3)
    for dtype, shape, K in ((torch.bfloat16, (2, 8, 3000, 128), 100), (torch.float32, (1, 3, 77, 128), 77),
                            (torch.float16, (3, 2, 500, 64), 1)):
        src = torch.randn(*shape, generator=g).to(dtype)
        idx = torch.randint(0, shape[2], (shape[0], shape[1], K), generator=g)
        want = torch.empty(shape[0], shape[1], K, shape[3], dtype=dtype)
        got = torch.full_like(want, 7)
        ref.gather_kv_out_cpu(src, idx, want)
        ext.gather_kv_out_cpu(src, idx, got)
        assert torch.equal(got.view(torch.uint8), want.view(torch.uint8))
        for b in range(shape[0]):
            for h in range(shape[1]):
                rows = O.gather_rows(src[b, h].view(torch.uint8).numpy(), idx[b, h].numpy())
                assert np.array_equal(rows, want[b, h].view(torch.uint8).numpy())
    # rows that are not contiguous, and an output that is a slice of a larger buffer
    src_t = torch.randn(2, 3, 128, 50, generator=g).transpose(2, 3)
    idx = torch.randint(0, 50, (2, 3, 9), generator=g)
    big_w, big_g = torch.zeros(2, 3, 20, 128), torch.zeros(2, 3, 20, 128)
    ref.gather_kv_out_cpu(src_t, idx, big_w[:, :, 4:13])
    ext.gather_kv_out_cpu(src_t, idx, big_g[:, :, 4:13])
    assert torch.equal(big_g, big_w)
    idx[1, 2, 8] = -1
    with pytest.raises(RuntimeError, match="out of bounds"):
        ref.gather_kv_out_cpu(src_t, idx, big_w[:, :, 4:13])
    with pytest.raises(RuntimeError, match="out of bounds"):
        ext.gather_kv_out_cpu(src_t, idx, big_g[:, :, 4:13])


def test_prefill_store_refuses_operands_of_several_devices():
    """The launch goes to the stream of k's device: rows, index or norms on another one are refused before it (host tensors
    that say they are on a GPU stand in for two cards)."""
    import torch

    from pariskv_amd import ops

    class On:
        def __init__(self, device, t):
            self._t, self.device, self.is_cuda = t, torch.device(device), True

        def get_device(self):
            return self.device.index

        def __getattr__(self, name):
            return getattr(self._t, name)

    def operands(**elsewhere):
        t = dict(k=torch.zeros(1, 2, 8, 128), v=torch.zeros(1, 2, 8, 128), signs=torch.ones(128), dk=torch.zeros(1, 2, 4, 128),
                 dv=torch.zeros(1, 2, 4, 128), zk=torch.zeros(1, 2, 5, 128), zv=torch.zeros(1, 2, 5, 128),
                 cb=torch.zeros(1, 2, 16, 5, dtype=torch.uint8), k4=torch.zeros(1, 2, 16, 5, 4, dtype=torch.uint8),
                 kw=torch.zeros(1, 2, 16, 5, dtype=torch.bfloat16), cc=torch.zeros(1, 2, 16, 256, dtype=torch.int32),
                 dn=torch.zeros(1, 2, 4), zn=torch.zeros(1, 2, 5), zn2=torch.zeros(1, 2, 5))
        return {n: On(elsewhere.get(n, "cuda:0"), x) for n, x in t.items()}

    for name in operands():
        o = operands(**{name: "cuda:1"})
        with pytest.raises(RuntimeError, match="tensors of one launch"):
            ops.prefill_store(o["k"], o["v"], 2, 5, o["signs"], (o["dk"], o["dv"]), 3, (o["zk"], o["zv"]),
                              (o["cb"], o["k4"], o["kw"], o["cc"]), dense_vnorm=o["dn"], zone_vnorm=o["zn"], zone_vnorm2=o["zn2"])


def test_prefill_store_has_room_for_the_longest_rows():
    """Token counts up to 2^29 pass the check of pkv_prefill_store (the index itself takes 2^24 keys a row); no kernel is
    launched, as there is no K/V to copy."""
    from pariskv_amd import _lib

    L = _lib.lib()
    a = _lib.PrefillArgs()
    a.dtype, a.bs, a.n_kv_heads, a.n_sink, a.n_tail, a.tail_row0 = _lib.DTYPE_BF16, 1, 1, 64, 512, 64
    for n, ok in ((1 << 23, True), ((1 << 24) + 5, True), ((1 << 29) - 577, True), ((1 << 29) - 576, False), (1 << 40, False), (-1, False)):
        a.n_encode = n
        assert L.pkv_prefill_store(a, None) == _lib.EINVAL
        assert (b"token counts" not in L.pkv_last_error()) == ok, (n, L.pkv_last_error())


def test_noalloc_scratch_takes_the_shapes_of_the_largest_chunks():
    """Rows scanned in chunks below 2048 keys need more room for histograms: near the end of the fixed scratch array such a shape
    is scanned in larger chunks instead of being refused.  (Shapes that the check lets through end at the null pointers.)"""
    from pariskv_amd import _lib

    L = _lib.lib()
    room = L.pkv_retrieve_noalloc_max_bytes()
    for rows, n, c, ok in ((93, 11158, 11158, True), (112, 8811, 8722, True), (8, 4096, 2048, True), (94, 11258, 11258, False),
                           (114, 8911, 8822, False)):
        a = _lib.RetrieveArgs()
        a.dtype, a.bs, a.n_kv_heads, a.group, a.n_keys, a.n_cand, a.k, a.cap, a.out_ids = _lib.DTYPE_BF16, 1, rows, 1, n, c, min(c, 8192), n, 256
        assert (L.pkv_retrieve_noalloc(a, None) != _lib.ENOMEM) == ok, (rows, n, c, L.pkv_retrieve_ws_bytes(rows, n, c, min(c, 8192)), room)


def test_one_chunk_rule():
    """ops.pick_chunk_keys (stand-alone scans) is the rule the retrieval lays its workspace out by: a row's histogram table
    there holds one entry a chunk, or four where chunks of 8192 keys and more are scanned in pieces."""
    from pariskv_amd import _lib, ops

    L = _lib.lib()
    for rows in (1, 2, 3, 8, 12, 64, 200, 1500):
        for n in (1, 255, 256, 257, 4000, 8192, 8193, 16385, 33000, 131072, 1000003, 1 << 24):
            chunk = ops.pick_chunk_keys(rows, n)
            n_chunks = -(-n // chunk)
            ptr, nbytes = ctypes.c_void_p(), ctypes.c_size_t()
            _lib.check(L.pkv_retrieve_ws_view(256, rows, n, n, 1, b"chunk_suffix_hist", ctypes.byref(ptr), ctypes.byref(nbytes)))
            pieces = 4 if chunk >= 8192 and 4 * n_chunks <= 512 else 1
            assert nbytes.value == rows * n_chunks * pieces * 256, (rows, n, chunk)


def _in_place_step(bs=1, H=8, group=4, n_keys=4096, n_cand=1500, k=100, sink=64, tail=529):
    """Argument blocks of a bf16 decode step that attends to the selected rows in place, with buffers side by side at made-up
    addresses: (retrieve, retrieval workspace and its bytes, attention)."""
    from pariskv_amd import _lib

    L = _lib.lib()
    a, aa, at = _lib.RetrieveArgs(), _lib.AttnArgs(), 1 << 32

    def take(nbytes):
        nonlocal at
        p, at = at, at + (nbytes + 255) // 256 * 256
        return p

    rows = bs * H
    a.dtype, a.bs, a.n_kv_heads, a.group, a.cap, a.n_keys, a.n_cand, a.k = _lib.DTYPE_BF16, bs, H, group, n_keys, n_keys, n_cand, k
    a.any_order, a.n_tiers = 1, 6
    a.q, a.out_ids, a.out_scores = take(rows * group * 256), take(rows * k * 8), take(rows * k * 4)
    ws_bytes = L.pkv_retrieve_ws_bytes(rows, n_keys, n_cand, k)
    ws = take(ws_bytes)
    total = sink + n_keys + tail
    K, V = take(rows * total * 256), take(rows * total * 256)
    for i, (row0, n, idx) in enumerate([(0, sink, 0), (sink, k, a.out_ids), (sink + n_keys, tail, 0)]):
        aa.segments[i] = _lib.AttnSegment(K, V, H * total * 128, total * 128, row0, n, idx or None, k if idx else 0, n_keys if idx else 0)
    aa.n_segments, aa.scale, aa.out = 3, 0.1, take(rows * group * 256)
    aa.ws_bytes = L.pkv_decode_attention_ws_bytes(bs, H, group, sink + k + tail)
    aa.ws = take(aa.ws_bytes)
    return a, ws, ws_bytes, aa


def test_decode_step_waits_where_buffers_are_shared():
    """pkv_decode_step is the retrieval followed by the attention: scratch memory, queries and results may be shared as that order
    allows.  The attention in two parts writes while the retrieval still works, so it is not taken there."""
    from pariskv_amd import _lib

    form = _lib.lib().pkv_decode_step_form
    for shape in ({}, dict(k=512), dict(n_keys=100000, n_cand=10000)):
        a, ws, ws_bytes, aa = _in_place_step(**shape)
        apart, at_ws, out = form(a, ws, aa), aa.ws, aa.out
        assert apart == (2 if shape.get("k") == 512 else 1)
        for p in (ws, ws + 256, ws + ws_bytes - 256, ws - 256, a.out_ids, a.out_scores, a.q):
            aa.ws = p
            assert form(a, ws, aa) == 0, (shape, p)
        aa.ws = at_ws
        for p in (ws, ws + ws_bytes - 256, a.out_ids, a.out_scores, a.q + 256, at_ws):
            aa.out = p
            assert form(a, ws, aa) == 0, (shape, p)
        aa.out = a.q  # in place of the queries: row by row
        assert form(a, ws, aa) == apart
        aa.out = out
        aa.ws = ws + ws_bytes  # right behind it
        assert form(a, ws, aa) == apart
        assert form(a, at_ws + aa.ws_bytes, aa) == apart


def test_decode_step_selects_several_times_a_row_only_in_one_round():
    """Several workgroups a row select the same keys each: where they are more than the chip takes at once, only if the rounds fill."""
    from pariskv_amd import _lib

    form = _lib.lib().pkv_decode_step_form
    for rows, cand, k, want in ((64, 8192, 1024, 2), (85, 8192, 1024, 2), (86, 8192, 1024, 0), (128, 8192, 700, 2), (129, 8192, 700, 0),
                                (192, 4097, 512, 0), (192, 4096, 512, 2), (96, 3000, 1024, 0), (96, 3000, 700, 2), (136, 1500, 700, 0),
                                (160, 3000, 1024, 2), (192, 3000, 1024, 0), (256, 4096, 512, 2), (256, 8192, 250, 1), (512, 1500, 200, 1)):
        a, ws, _, aa = _in_place_step(bs=rows, H=1, n_keys=20000, n_cand=cand, k=k)
        assert form(a, ws, aa) == want, (rows, cand, k)


def test_decode_step_merges_up_to_six_blocks_in_one_workgroup():
    """Selected keys in up to six blocks of 32 are one workgroup's; beyond, several workgroups' where they fit one round and the
    selection is one launch."""
    from pariskv_amd import _lib

    form = _lib.lib().pkv_decode_step_form
    for rows, cand, k, want in ((8, 4000, 160, 1), (8, 4000, 192, 1), (8, 4000, 193, 2), (64, 4000, 192, 1), (8, 9000, 192, 1),
                                (8, 9000, 193, 0), (8, 9000, 512, 0), (128, 9000, 250, 1), (128, 9000, 257, 0), (8, 4000, 1024, 2), (8, 4000, 1025, 0)):
        a, ws, _, aa = _in_place_step(bs=rows, H=1, n_keys=20000, n_cand=cand, k=k)  # 64 rows before the selected ones: two whole blocks
        assert form(a, ws, aa) == want, (rows, cand, k)


def test_topk_kernels_have_no_scratch(tmp_path):
    """The selections hold up to 32 scores a thread in the 128 registers that 16 waves a CU leave: a spilled one is a trip to memory."""
    from pariskv_amd import _lib

    llvm = "/opt/rocm/llvm/bin/"
    if not (os.path.exists(llvm + "llvm-objdump") and os.path.exists(llvm + "llvm-readelf")):
        pytest.skip("no tools to read the library")
    if not os.path.exists(_lib.SO_PATH):
        _lib.build()
    shutil.copy(_lib.SO_PATH, tmp_path / "lib.so")   # the parts are written beside it
    subprocess.run([llvm + "llvm-objdump", "--offloading", "lib.so"], cwd=tmp_path, check=True, capture_output=True)
    sizes = {}
    for part in tmp_path.glob("lib.so.*gfx950"):
        notes = subprocess.run([llvm + "llvm-readelf", "--notes", str(part)], check=True, capture_output=True, text=True).stdout
        for kernel in re.split(r"(?m)^  - ", notes):
            name, size = re.search(r"(?m)^    \.name: +(\S+)", kernel), re.search(r"\.private_segment_fixed_size: +(\d+)", kernel)
            if name and size:
                sizes[name.group(1)] = int(size.group(1))
    topk = {n: s for n, s in sizes.items() if "pkv_topk" in n}
    assert sum("long" in n for n in topk) == 4 and not any(topk.values()), topk
