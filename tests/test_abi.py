"""The C ABI: the library loads, exports every entry point include/qwen_state.h declares, and rejects bad
arguments with QS_EINVAL before any launch (no GPU needed); the Python ops validate before calling."""
import ctypes
import os
import re

import pytest
import torch

import qwen36_state as Q
from qwen36_state import _lib, ops

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include", "qwen_state.h")
FAKE = ctypes.c_void_p(0x1000)  # never dereferenced: every call below fails validation first
NUL = ctypes.c_void_p(0)
S = ctypes.c_void_p(0)


def declared():
    text = open(HEADER).read()
    return sorted(set(re.findall(r"\b(qs_\w+)\s*\(", text)))


def test_exports_every_declared_symbol():
    L = Q.lib()
    names = declared()
    assert len(names) >= 14
    for n in names:
        assert hasattr(L, n), n
        assert n in _lib.SIGNATURES, n
    assert set(_lib.SIGNATURES) == set(names)
    assert L.qs_abi_version() == 4


def test_rejects_bad_arguments():
    L = Q.lib()
    # null pointer
    assert L.qs_gdn_decode_step(NUL, FAKE, FAKE, FAKE, FAKE, FAKE, FAKE, 1, 16, 48, 128, 128, 0.1, 1e-6, S) == -1
    assert "null" in L.qs_last_error().decode()
    # unsupported head dims / grouping
    assert L.qs_gdn_decode_step(FAKE, FAKE, FAKE, FAKE, FAKE, FAKE, FAKE, 1, 16, 48, 64, 128, 0.1, 1e-6, S) == -1
    assert L.qs_gdn_decode_step(FAKE, FAKE, FAKE, FAKE, FAKE, FAKE, FAKE, 1, 16, 40, 128, 128, 0.1, 1e-6, S) == -1
    assert "multiple" in L.qs_last_error().decode()
    assert L.qs_conv1d_update(FAKE, FAKE, FAKE, FAKE, 1, 10240, 3, S) == -1
    assert L.qs_gdn_verify_step(FAKE, FAKE, FAKE, FAKE, FAKE, FAKE, FAKE, FAKE, FAKE, NUL, NUL,
                                1, 9, 16, 48, 128, 128, 4, 0.1, 1e-6, S) == -1  # fmt: skip
    assert L.qs_gdn_verify_step(FAKE, FAKE, FAKE, FAKE, FAKE, FAKE, FAKE, FAKE, FAKE, NUL, NUL,
                                1, 4, 16, 48, 128, 128, 4, 0.1, 1e-6, S) == -1  # fmt: skip  (states_out aliases)
    assert "alias" in L.qs_last_error().decode()
    # attention: head dim, block size, group size, missing workspace
    args = lambda hd, blk, nq, mb, pps, ws: (FAKE, NUL, NUL, FAKE, FAKE, FAKE, FAKE, FAKE, ws, 1, 1, nq, 4, hd, blk,
                                             mb, 2048, pps, 0.0625, NUL, S)  # fmt: skip
    assert L.qs_paged_gqa_decode(*args(128, 64, 24, 512, 8, FAKE)) == -1
    assert L.qs_paged_gqa_decode(*args(256, 32, 24, 512, 8, FAKE)) == -1
    assert L.qs_paged_gqa_decode(*args(256, 64, 20, 512, 8, FAKE)) == -1
    assert L.qs_paged_gqa_decode(*args(256, 64, 24, 512, 8, NUL)) == -1
    assert "workspace" in L.qs_last_error().decode()
    # fill: a table too short for the tokens
    assert L.qs_paged_kv_fill(FAKE, FAKE, FAKE, FAKE, FAKE, 200, 0, 4, 256, 64, 3, 2048, S) == -1
    assert L.qs_paged_kv_append(FAKE, FAKE, FAKE, FAKE, FAKE, FAKE, 1, 1, 4, 250, 64, 8, 8, NUL, S) == -1
    # the length advance: null lengths, aliasing base
    assert L.qs_advance_lengths(NUL, NUL, 4, 1, 4096, NUL, S) == -1
    assert L.qs_advance_lengths(FAKE, FAKE, 4, 1, 4096, NUL, S) == -1
    assert "alias" in L.qs_last_error().decode()
    # gather: a table too short for the positions, a pool without its output
    assert L.qs_paged_kv_gather(FAKE, FAKE, FAKE, FAKE, FAKE, 200, 0, 4, 256, 64, 3, 2048, S) == -1
    assert L.qs_paged_kv_gather(FAKE, FAKE, FAKE, NUL, FAKE, 100, 0, 4, 256, 64, 3, 2048, S) == -1
    # prompt conv: taps, ldx below C or not a multiple of 8, CQ not a multiple of 8, misalignment, null x
    conv = lambda x, ldx, T, cq, k: (x, ldx, NUL, FAKE, FAKE, FAKE, FAKE, FAKE, T, cq, 6144, k, S)
    assert L.qs_conv1d_prefill(*conv(FAKE, 10240, 5, 2048, 3)) == -1
    assert L.qs_conv1d_prefill(*conv(FAKE, 10000, 5, 2048, 4)) == -1
    assert L.qs_conv1d_prefill(*conv(FAKE, 10244, 5, 2048, 4)) == -1
    assert L.qs_conv1d_prefill(*conv(FAKE, 10240, 5, 2044, 4)) == -1
    assert L.qs_conv1d_prefill(*conv(ctypes.c_void_p(0x1008), 10240, 5, 2048, 4)) == -1
    assert "aligned" in L.qs_last_error().decode()
    assert L.qs_conv1d_prefill(*conv(NUL, 10240, 5, 2048, 4)) == -1
    assert "null" in L.qs_last_error().decode()


def test_workspace_sizes():
    L = Q.lib()
    assert L.qs_gdn_workspace_bytes(8, 16) == 8 * 16 * 2 * 4
    one = L.qs_paged_attention_workspace_bytes(1, 1, 24, 4, 256, 512, 8)
    assert one > 64 * 4 * 6 * 256 * 4  # at least the level-0 partials of 64 splits
    assert L.qs_paged_attention_workspace_bytes(1, 1, 24, 4, 128, 512, 8) == 0


def test_attention_workspace_serves_smaller_calls():
    """A workspace sized for a call holds the partials of every call of fewer users, tokens or table entries, though a
    smaller grid is cut into more splits."""
    size = lambda B, T, mb, pps: Q.lib().qs_paged_attention_workspace_bytes(B, T, 24, 4, 256, mb, pps)  # noqa: E731
    for pps in (1, 2, 8, 16, 64):
        for T in (1, 4, 16):
            for B in (1, 3, 8, 70):
                for mb in (1, 7, 64, 500):
                    whole = size(B, T, mb, pps)
                    assert all(size(b, t, m, pps) <= whole
                               for b in (1, B // 2 + 1, B) for t in (1, T) for m in (1, mb // 3 + 1, mb) if b <= B and m <= mb)  # fmt: skip


def test_attention_walk_pages():
    """The grain suggested for a call: never more pages than the caller's, its partials fit a workspace sized at the
    caller's grain (and so do the plain call's and the mixer's), and arguments the launch refuses come back as they are."""
    L = Q.lib()
    for pps in (1, 2, 8, 16, 64):
        for T in (1, 2, 3, 4, 8, 11, 16):
            for B in (1, 3, 8, 33, 70, 300):
                for mb in (1, 2, 3, 4, 5, 7, 64, 500):
                    rows = T * 6
                    size = L.qs_paged_attention_workspace_bytes(B, T, 24, 4, 256, mb, pps)
                    for mixer in (0, 1):
                        walk = L.qs_paged_attention_walk_pages(B, T, 24, 4, mb, pps, mixer)
                        assert 1 <= walk <= pps
                        parts = B * 4 * -(-mb // walk) * rows
                        assert 65536 + -(-parts * 8 // 256) * 256 + parts * 1024 <= size
    for pps, mb, nq in ((0, 64, 24), (-3, 64, 24), (65, 64, 24), (1, 1025, 24), (8, 64, 23), (8, 0, 24)):
        assert L.qs_paged_attention_walk_pages(1, 1, nq, 4, mb, pps, 0) == pps


@pytest.mark.parametrize("name,raw", [("cuda:0", False), ("cuda", True)])
def test_stream_handle_falls_back_to_the_public_call(monkeypatch, name, raw):
    """A torch without the raw stream call, or a device without an index: the stream object's handle."""
    class Stream:
        cuda_stream = 77

    monkeypatch.setattr(torch.cuda, "current_stream", lambda dev: Stream)
    monkeypatch.setattr(ops, "_raw_stream", (lambda index: 1 + index) if raw else None)
    assert ops._stream(torch.device(name)) == 77


def test_ops_validate_before_calling():
    cpu = torch.zeros(1, 16, 128, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="GPU"):
        ops.gdn_decode_step(cpu, cpu, torch.zeros(1, 48, 128, dtype=torch.bfloat16), torch.zeros(1, 48),
                            torch.zeros(1, 48), torch.zeros(1, 48, 128, 128))  # fmt: skip
    with pytest.raises(ValueError):
        ops.paged_gqa_decode(torch.zeros(1, 1, 24, 256), torch.zeros(8, 4, 64, 256), torch.zeros(8, 4, 64, 256),
                             torch.zeros(1, 8, dtype=torch.int32), torch.zeros(1, dtype=torch.int32), 0.0625)  # fmt: skip
