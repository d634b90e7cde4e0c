"""The weights' row-pair copies are prepared weights: made once per weight, held by the weight
tensor itself, made only where the GEMM reads them.  CPU-side: the C queries (no device work) and
the caching logic with the pack counted (pack_row_pairs replaced by a counting stand-in)."""
import pytest
import torch

from lockstep_amd import _lib as L
from lockstep_amd import ops


def test_gemm_row_pair_query():
    lib = L.load()
    # one activation row streams W8 whole rows; mid row counts read whole lines of W8 a K stage: no copy
    for M in (1, 4, 64, 128):
        assert lib.lsk_gemm_reads_row_pairs(M, 28672, 4096) == 0, M
    # decode rows of wide weights whose activations fit in LDS: the skinny GEMV streams the copy
    for M, N, K in ((8, 28672, 4096), (32, 28672, 4096), (16, 14336, 4096)):
        assert lib.lsk_gemm_reads_row_pairs(M, N, K) == 1, (M, N, K)
    # narrow weights stream whole rows through LDS; 32 rows of K = 14336 exceed the LDS
    for M, N, K in ((16, 3584, 3584), (8, 4096, 14336), (32, 16384, 14336)):
        assert lib.lsk_gemm_reads_row_pairs(M, N, K) == 0, (M, N, K)
    # prefill row counts on the ping-pong tiles read it
    for M, N, K in ((2048, 28672, 4096), (2048, 4096, 14336), (8192, 37888, 3584), (8192, 3584, 18944)):
        assert lib.lsk_gemm_reads_row_pairs(M, N, K) == 1, (M, N, K)
    assert lib.lsk_gemm_reads_row_pairs(2048, 4096, 100) == 0        # K % 16 != 0
    assert lib.lsk_gemm_reads_row_pairs(0, 4096, 4096) == 0


def test_moe_row_pair_query():
    lib = L.load()
    E, k, H, I = 128, 8, 2048, 768
    assert lib.lsk_moe_reads_row_pairs(1, k, E, H, I, 0, 0) == 0       # the grouped GEMV
    for T in (2, 32, 192):                                                 # the skinny grouped GEMM
        assert lib.lsk_moe_reads_row_pairs(T, k, E, H, I, 0, 0) == 1, T
    assert lib.lsk_moe_reads_row_pairs(4096, k, E, H, I, 0, 0) == 1    # the ping-pong tiles
    assert lib.lsk_moe_reads_row_pairs(32, k, E, H, I, 8, 0) == 0      # rotated layers: the tiles
    # a per-call choice of the register-staged tile or the GEMV (select = variant + 2) reads none
    assert lib.lsk_moe_reads_row_pairs(4096, k, E, H, I, 0, 2) == 0
    assert lib.lsk_moe_reads_row_pairs(32, k, E, H, I, 0, 4) == 0
    # the thread's own setting is left as it was
    assert lib.lsk_moe_reads_row_pairs(4096, k, E, H, I, 0, 0) == 1


def test_moe_mx_skinny_query():
    """MXFP4 layers (GPT-OSS-20B: E 32, top 4, H = I = 2880, 90 E8M0 bytes a row) read the codes'
    skinny-layout copies from 1 to 256 tokens (one token only when k * 2I / 64 >= 320: with top 2
    the MX GEMV keeps it); under lsk_moe_mx_select(3) from one token; forced kernel families read
    none."""
    lib = L.load()
    E, k, H, I, lds = 32, 4, 2880, 2880, 90
    assert lib.lsk_moe_mx_reads_skinny(1, 2, E, H, I, lds, lds, 0, 0) == 0            # the MX GEMV
    assert lib.lsk_moe_mx_reads_skinny(1, 2, E, H, I, lds, lds, 0, 4) == 1            # mx_select 3
    for T in (1, 2, 24, 25, 128, 256):
        assert lib.lsk_moe_mx_reads_skinny(T, k, E, H, I, lds, lds, 0, 0) == 1, T
    for T in (257, 4096):                                                             # the tiles
        assert lib.lsk_moe_mx_reads_skinny(T, k, E, H, I, lds, lds, 0, 0) == 0, T
    assert lib.lsk_moe_mx_reads_skinny(1, k, E, H, I, lds, lds, 0, 4) == 1            # mx_select 3
    assert lib.lsk_moe_mx_reads_skinny(200, k, E, H, I, lds, lds, 2, 4) == 1          # ... over the tiles
    # a forced kernel family (select = variant + 2) reads none; the thread's settings stay as they were
    assert lib.lsk_moe_mx_reads_skinny(32, k, E, H, I, lds, lds, 2, 0) == 0
    assert lib.lsk_moe_mx_reads_skinny(32, k, E, H, I, lds, lds, 4, 4) == 0           # the GEMV forced
    assert lib.lsk_moe_mx_reads_skinny(32, k, E, H, I, lds, lds, 0, 2) == 0           # mx_select 1
    assert lib.lsk_moe_mx_reads_skinny(32, k, E, H, I, lds, lds, 0, 0) == 1
    # the chunk's rows and the E8M0 rows must fit the LDS: K = 16384 does not
    assert lib.lsk_moe_mx_reads_skinny(32, k, E, 16384, I, 512, lds, 0, 0) == 0
    assert lib.lsk_moe_mx_reads_skinny(32, k, E, H, I, lds, lds, 0, 10) == 0          # out of range
    # the grouped linear alone: experts averaging at most 32 rows
    assert lib.lsk_grouped_mx_reads_skinny(256, E, H, lds) == 1
    assert lib.lsk_grouped_mx_reads_skinny(32 * E, E, H, lds) == 1
    assert lib.lsk_grouped_mx_reads_skinny(32 * E + 1, E, H, lds) == 0
    assert lib.lsk_grouped_mx_reads_skinny(256, E, 16384, 512) == 0
    assert lib.lsk_grouped_mx_reads_skinny(256, E, 100, 4) == 0                        # K % 32 != 0


def test_mx_skinny_copy_size_and_argument_checks():
    """lsk_mx_skinny_bytes: 1 KB per group of 16 rows and step of 4 blocks (partial ones whole); the
    pack refuses K % 32 != 0, a row stride below K / 2 or not a multiple of 4, and null pointers,
    before any device work."""
    lib = L.load()
    assert lib.lsk_mx_skinny_bytes(16, 128) == 1024
    assert lib.lsk_mx_skinny_bytes(17, 128) == 2048
    assert lib.lsk_mx_skinny_bytes(16, 160) == 2048            # 5 blocks: two steps
    assert lib.lsk_mx_skinny_bytes(5760, 2880) == 360 * 23 * 1024
    for args in ((64, 16, 40), (16, 16, 64), (34, 16, 64)):     # (ldw, rows, K)
        ldw, rows, K = args
        assert lib.lsk_mx_skinny_pack(16, ldw, rows, K, 4096, None) != 0, args
    assert lib.lsk_mx_skinny_pack(None, 64, 16, 64, 4096, None) != 0
    assert "lsk_mx_skinny_pack" in L.last_error()


@pytest.fixture
def counting_pack(monkeypatch):
    made = []

    def fake_pack(w):
        made.append((w.data_ptr(), tuple(w.shape)))
        return torch.empty((L.load().lsk_row_pairs_bytes(*w.shape),), dtype=torch.int8)
    monkeypatch.setattr(ops, "pack_row_pairs", fake_pack)
    return made


def test_130_dense_weights_pack_once(counting_pack):
    """A model's worth of distinct dense weights (130) cycled twice through the prefill path: each
    copy is made on the first pass and reused on the second (decode rows that read it share the same
    copy); one activation row makes none."""
    ws = [torch.zeros((8192, 64), dtype=torch.int8) for _ in range(130)]
    for w in ws:
        assert ops.row_pairs_of(w, 1) is None
    assert counting_pack == []
    first = [ops.row_pairs_of(w, 2048) for w in ws]
    assert len(counting_pack) == 130 and all(p is not None for p in first)
    second = [ops.row_pairs_of(w, 2048) for w in ws]
    assert len(counting_pack) == 130
    assert all(a is b for a, b in zip(first, second))
    assert all(ops.row_pairs_of(w, 32) is p for w, p in zip(ws, first)) and len(counting_pack) == 130
    # views of the same storage (the reference's b8 = W8.t() turned back) share the copy
    assert ops.row_pairs_of(ws[0].t().t(), 2048) is first[0]
    # an in-place update re-makes that weight's copy only
    ws[7].add_(1)
    assert ops.row_pairs_of(ws[7], 2048) is not first[7]
    assert len(counting_pack) == 131
    assert ops.row_pairs_of(ws[8], 2048) is first[8] and len(counting_pack) == 131


def test_copy_lives_with_the_weight(counting_pack):
    import gc
    import weakref
    w = torch.zeros((64, 64), dtype=torch.int8)
    p = ops.row_pairs_of(w, 4096)
    ref = weakref.ref(p)
    del p
    assert ref() is not None                 # held by the weight
    ops.release_row_pairs(w)
    gc.collect()
    assert ref() is None
    p = ops.row_pairs_of(w, 4096)
    ref = weakref.ref(p)
    del p, w
    gc.collect()
    assert ref() is None                     # freed with the weight


def test_copies_can_be_turned_off(counting_pack, monkeypatch):
    monkeypatch.setattr(ops, "ROW_PAIR_COPIES", False)
    assert ops.row_pairs_of(torch.zeros((64, 64), dtype=torch.int8), 4096) is None
    assert counting_pack == []


def test_copy_on_another_stream_waits_for_the_pack(monkeypatch):
    """The copy's pack is ordered on the stream of the call that makes it: another stream's first use
    waits for the event after it and marks the copy as used there, once; the making stream does neither."""
    log = []

    class Stream:
        def __init__(self, handle):
            self.cuda_stream = handle

        def wait_event(self, event):
            log.append(("wait", self.cuda_stream, event.at))

    class Event:
        def record(self, stream):
            self.at = stream.cuda_stream

    class Copy:
        is_cuda, device = True, "dev"

        def record_stream(self, stream):
            log.append(("used", stream.cuda_stream))

    now = [Stream(1)]
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: now[0])
    monkeypatch.setattr(torch.cuda, "Event", Event)
    monkeypatch.setattr(L, "stream_of", lambda t: now[0].cuda_stream)
    copy = Copy()
    held = ops._RowPairs(0, copy)
    ops._packed_on_current_stream([held])
    assert held.on_current_stream() is copy and log == []
    now[0] = Stream(2)
    for _ in range(2):
        assert held.on_current_stream() is copy and log == [("wait", 2, 1), ("used", 2)]
    now[0] = Stream(1)
    assert held.on_current_stream() is copy and len(log) == 2


def test_an_expert_list_shares_one_event(counting_pack, monkeypatch):
    """The copies of a list of weights are stored with one event, recorded once behind all their packs."""
    calls = []
    monkeypatch.setattr(ops, "_packed_on_current_stream", lambda made: calls.append((len(counting_pack), len(made))))
    ws = [torch.zeros((64, 64), dtype=torch.int8) for _ in range(5)]
    copies = ops.row_pair_copies(ws)
    assert calls == [(5, 5)] and all(c is ops.row_pairs_of(w, 4096) for c, w in zip(copies, ws))
    ws[2].add_(1)
    again = ops.row_pair_copies(ws)
    assert [a is c for a, c in zip(again, copies)] == [True, True, False, True, True] and (6, 1) in calls


def test_weights_with_copies_save_and_deepcopy(counting_pack, tmp_path):
    """A weight that holds a copy is saved, loaded (weights_only) and deep-copied as before, without the
    copy, which its own first use makes."""
    import copy
    w = torch.arange(64 * 64).view(64, 64).to(torch.int8)
    first = ops.row_pairs_of(w, 4096)
    torch.save(w, tmp_path / "w.pt")
    for t in (torch.load(tmp_path / "w.pt", weights_only=True), copy.deepcopy(w)):
        assert torch.equal(t, w)
        assert ops.row_pairs_of(t, 4096) is not first and ops.row_pairs_of(t, 4096) is ops.row_pairs_of(t, 4096)
    assert ops.row_pairs_of(w, 4096) is first and len(counting_pack) == 3


def test_inference_tensors_go_without_copies(counting_pack):
    """A weight made under inference mode has no version counter: the GEMMs read it itself, in and out of
    that mode.  An ordinary weight keeps its copy under inference mode, and in-place writes made there
    still make it stale."""
    with torch.inference_mode():
        w = torch.zeros((64, 64), dtype=torch.int8)
        assert ops.row_pairs_of(w, 4096) is None
    assert ops.row_pairs_of(w, 4096) is None and counting_pack == []
    w = torch.zeros((64, 64), dtype=torch.int8)
    first = ops.row_pairs_of(w, 4096)
    with torch.inference_mode():
        assert ops.row_pairs_of(w.t().t(), 4096) is first
        w.add_(1)
        assert ops.row_pairs_of(w, 4096) is not first
    assert len(counting_pack) == 2


def test_head_planes_pack_in_prepare_only(counting_pack):
    """A wide head's planes get their copy where prepare asks for it (some decode batch reads it); calls
    read that copy, or the planes after an in-place update, and never pack.  Narrow heads get none."""
    w2 = torch.zeros((2 * 8200, 272), dtype=torch.int8)
    assert ops.planes_pairs(w2, 8, 15) is None and counting_pack == []
    ops.prepare_planes_pairs(w2, 15)
    assert len(counting_pack) == 1
    for rows, abits, reads in ((3, 15, True), (16, 15, True), (17, 15, False), (0, 15, False), (1, 8, False),
                               (32, 8, True), (33, 8, False)):
        assert (ops.planes_pairs(w2, rows, abits) is not None) == reads, (rows, abits)
    w2.add_(1)
    assert ops.planes_pairs(w2, 8, 15) is None and len(counting_pack) == 1
    ops.prepare_planes_pairs(w2, 15)
    assert ops.planes_pairs(w2, 8, 15) is not None and len(counting_pack) == 2
    for narrow in (torch.zeros((512, 272), dtype=torch.int8), torch.zeros((16400, 40), dtype=torch.int8)):
        ops.prepare_planes_pairs(narrow, 15)
    assert len(counting_pack) == 2


def test_head_planes_without_room_for_the_copy(monkeypatch):
    """A device with no room for the planes' copy prepares the head without it."""
    def no_room(w):
        raise torch.OutOfMemoryError("no room")
    monkeypatch.setattr(ops, "pack_row_pairs", no_room)
    w2 = torch.zeros((16400, 64), dtype=torch.int8)
    ops.prepare_planes_pairs(w2, 15)
    assert ops.planes_pairs(w2, 8, 15) is None
