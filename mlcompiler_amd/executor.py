"""HipExecutor: the Python face of the C ABI, with the method names, argument
order and bool-return conventions of the reference's MetalExecutor paged path
(compiler/runtime/metal_runtime.hpp:181-183, 510-533, 619-703), so that tests
read like tests/test_paged_flash.cpp and tests/test_paged_kv.cpp.

Buffers are opaque device pointers (ints), metadata are sequences of uint32.
Nothing here computes: every method is one call into csrc/libmlc_hip.so, the ones of a program's
inner loop through the module _call (csrc/py_call.cpp), the others through ctypes.
"""
from __future__ import annotations

import ctypes as C

import numpy as np

from ._lib import NativeLibraryError, load

_u32p = C.POINTER(C.c_uint32)


def _u32(seq) -> np.ndarray:
    return np.ascontiguousarray(seq, dtype=np.uint32)


def _ptr(a: np.ndarray):
    return a.ctypes.data_as(_u32p)


class HipExecutor:
    """Singleton, like MetalExecutor::Instance() (metal_runtime.mm:5774-5777)."""

    _instance = None

    @classmethod
    def Instance(cls) -> "HipExecutor":
        if cls._instance is None:
            cls._instance = cls()
        return cls._instance

    def __init__(self):
        self._lib = load()
        from . import _call    # (built next to the library that load() has just checked)
        self._call = _call

    # -- availability / errors
    def isAvailable(self) -> bool:
        return bool(self._lib.mlc_hip_available())

    def requireAvailable(self) -> None:
        if not self.isAvailable():
            raise NativeLibraryError("no gfx950 device: " + self.lastError())

    def lastError(self) -> str:
        return self._lib.mlc_hip_last_error().decode()

    # -- buffers (metal_runtime.hpp:693-703)
    def allocateScratchBuffer(self, nbytes: int) -> int:
        return self._lib.mlc_hip_alloc(nbytes) or 0

    def releaseScratchBuffer(self, buffer: int) -> None:
        self._lib.mlc_hip_free(buffer)

    def getOrAllocCachedBuffer(self, name: str, nbytes: int) -> int:
        return self._lib.mlc_hip_cached(name.encode(), nbytes) or 0

    def uploadToBuffer(self, buffer: int, src: np.ndarray, nbytes: int | None = None,
                       dst_offset: int = 0) -> bool:
        src = np.ascontiguousarray(src)
        n = src.nbytes if nbytes is None else nbytes
        return bool(self._lib.mlc_hip_upload(buffer, src.ctypes.data, n, dst_offset))

    def downloadFromBuffer(self, buffer: int, dst: np.ndarray, nbytes: int | None = None,
                           src_offset: int = 0) -> bool:
        assert dst.flags.c_contiguous and dst.flags.writeable
        n = dst.nbytes if nbytes is None else nbytes
        return bool(self._lib.mlc_hip_download(buffer, dst.ctypes.data, n, src_offset))

    def zeroBuffer(self, buffer: int, nbytes: int) -> bool:
        return bool(self._lib.mlc_hip_zero(buffer, nbytes))

    # -- forward pass (metal_runtime.hpp:181-183)
    def beginForwardPassCB(self) -> bool:
        return self._call.begin()

    def flushForwardPassCB(self) -> bool:
        return self._call.flush()

    def hasForwardPassCB(self) -> bool:
        return bool(self._lib.mlc_hip_has_open_pass())

    # -- paged flash attention (metal_runtime.hpp:510-523, 645-658)
    def runPagedFlashAttention(self, q_buffer, k_pages_buffer, v_pages_buffer, o_buffer,
                               page_tables_flat, page_table_offsets, seq_lens, q_positions,
                               batch, num_heads, kv_heads, head_dim, page_size_tokens,
                               apply_causal) -> bool:
        return self._call.attention(q_buffer, k_pages_buffer, v_pages_buffer, o_buffer, page_tables_flat,
                                    page_table_offsets, seq_lens, q_positions, batch, num_heads, kv_heads,
                                    head_dim, page_size_tokens, apply_causal, True)

    def encodePagedFlashAttention(self, q_buf, k_pages_buf, v_pages_buf, o_buf, page_tables_flat,
                                  page_table_offsets, seq_lens, q_positions, batch, num_heads,
                                  kv_heads, head_dim, page_size_tokens, apply_causal) -> bool:
        return self._call.attention(q_buf, k_pages_buf, v_pages_buf, o_buf, page_tables_flat, page_table_offsets,
                                    seq_lens, q_positions, batch, num_heads, kv_heads, head_dim, page_size_tokens,
                                    apply_causal, False)

    # -- batched paged KV write (metal_runtime.hpp:526-533, 680-687)
    def scatterKVPagedBatched(self, page_storage_buffer, page_ids, slots_in_page,
                              page_size_tokens, n_kv_heads, head_dim, batch, src_buffer) -> bool:
        return self._call.scatter_batched(page_storage_buffer, page_ids, slots_in_page, page_size_tokens,
                                          n_kv_heads, head_dim, batch, src_buffer, True)

    def encodeScatterKVPagedBatched(self, page_storage_buffer, page_ids, slots_in_page,
                                    page_size_tokens, n_kv_heads, head_dim, batch,
                                    src_buffer) -> bool:
        return self._call.scatter_batched(page_storage_buffer, page_ids, slots_in_page, page_size_tokens,
                                          n_kv_heads, head_dim, batch, src_buffer, False)

    # -- single-request scatter / gather (metal_runtime.hpp:619-626, 666-674)
    def scatterKVPaged(self, page_storage_buffer, page_table, page_size_tokens, n_kv_heads,
                       head_dim, tokens, start_slot, src_buffer, dtype_bytes) -> bool:
        return self._call.scatter(page_storage_buffer, page_table, page_size_tokens, n_kv_heads, head_dim, tokens,
                                  start_slot, src_buffer, dtype_bytes)

    def gatherKVPages(self, page_storage_buffer, page_table, page_size_tokens, n_kv_heads,
                      head_dim, num_tokens, dst_buffer, dtype_bytes) -> bool:
        return self._call.gather(page_storage_buffer, page_table, page_size_tokens, n_kv_heads, head_dim, num_tokens,
                                 dst_buffer, dtype_bytes)

    # -- the step before the KV write (metal_runtime.hpp:540-547, metal_runtime.mm:7915-8025)
    def encodeQkvSplitRopeCast(self, qkv_buf, q_buf, k_buf, v_buf, k_f16_buf, v_f16_buf, cos_buf,
                               sin_buf, batch, num_heads, kv_heads, head_dim, qkv_rows, q_rows,
                               k_rows, v_rows, rotary_dim, sync: bool = False) -> bool:
        return self._call.rope_cast(
            qkv_buf, q_buf, k_buf, v_buf, k_f16_buf, v_f16_buf, cos_buf, sin_buf, batch, num_heads,
            kv_heads, head_dim, qkv_rows, q_rows, k_rows, v_rows, rotary_dim, sync)

    # the same step fused with the two batched scatters that follow it in the walker
    # (batched_walker.cpp:287-331); no single reference method
    def encodeQkvSplitRopeScatter(self, qkv_buf, q_buf, k_pages_buffer, v_pages_buffer, cos_buf,
                                  sin_buf, page_ids, slots_in_page, page_size_tokens, batch,
                                  num_heads, kv_heads, head_dim, qkv_rows, q_rows, k_rows, v_rows,
                                  rotary_dim, k_f32_buf=None, v_f32_buf=None,
                                  sync: bool = False) -> bool:
        ids = _u32(page_ids)
        sl = _u32(slots_in_page)
        if ids.size != batch or sl.size != batch:
            return False
        return bool(self._lib.mlc_hip_qkv_split_rope_scatter(
            qkv_buf, q_buf, k_pages_buffer, v_pages_buffer, k_f32_buf, v_f32_buf, cos_buf, sin_buf,
            _ptr(ids), _ptr(sl), page_size_tokens, batch, num_heads, kv_heads, head_dim, qkv_rows,
            q_rows, k_rows, v_rows, rotary_dim, int(bool(sync))))

    # -- the other per-layer operators of the batched decode step
    def encodeRmsNormBatched(self, in_buf, weight, epsilon, batch, length, out_buf,
                             sync: bool = False) -> bool:  # metal_runtime.hpp:474-479
        return self._call.rms_norm(in_buf, weight, epsilon, batch, length, out_buf, sync)

    def encodeAddBatched(self, a_buf, b_buf, out_buf, total_elements, sync: bool = False) -> bool:
        return self._call.add(a_buf, b_buf, out_buf, total_elements, sync)  # metal_runtime.hpp:501-502

    def encodeSiluMulBatched(self, gate_buf, up_buf, out_buf, total_elements,
                             sync: bool = False) -> bool:  # metal_runtime.hpp:505-506
        return bool(self._lib.mlc_hip_silu_mul_batched(gate_buf, up_buf, out_buf, total_elements,
                                                       int(bool(sync))))

    def encodeGateUpSplitSiluMul(self, gate_up_buf, gate_buf, up_buf, out_buf, batch, ffn_inner,
                                 ffn_gate_up_rows, sync: bool = False) -> bool:  # :549-552
        return self._call.gate_up(gate_up_buf, gate_buf, up_buf, out_buf, batch, ffn_inner, ffn_gate_up_rows, sync)

    def encodeMatMulQ4_0Batched(self, weight_name, weights, in_buf, batch, rows, cols, row_stride,
                                quant_version, out_buf, sync: bool = False) -> bool:
        """metal_runtime.hpp:481-489; `weights` is the host byte array of the Q4_0 rows."""
        return self._call.matmul_q4_0(weight_name, weights, in_buf, batch, rows, cols, row_stride, quant_version,
                                      out_buf, sync)

    def encodeMatMulQ6KBatched(self, weight_name, weights, in_buf, batch, rows, cols, row_stride,
                               out_buf, sync: bool = False) -> bool:
        """metal_runtime.hpp:491-498 (sync=True: runMatMulQ6KBatched, :452-459); `weights` is the
        host byte array of the Q6_K rows."""
        return self._call.matmul_q6_k(weight_name, weights, in_buf, batch, rows, cols, row_stride, out_buf, sync)

    # -- chunked prefill (no reference method; see include/mlc_hip.h)
    def runPagedPrefillAttention(self, q_f16_buffer, k_pages_buffer, v_pages_buffer, o_buffer,
                                 page_tables_flat, page_table_offsets, seq_lens, q_start, batch,
                                 chunk, num_heads, kv_heads, head_dim, page_size_tokens,
                                 sync: bool = True) -> bool:
        return self._call.prefill(q_f16_buffer, k_pages_buffer, v_pages_buffer, o_buffer, page_tables_flat,
                                  page_table_offsets, seq_lens, q_start, batch, chunk, num_heads, kv_heads, head_dim,
                                  page_size_tokens, sync)

    # -- a pass replayed from a HIP graph
    def captureBegin(self) -> bool:
        return bool(self._lib.mlc_hip_capture_begin())

    def captureEnd(self) -> int:
        """Handle > 0 of the captured pass, or 0 (see lastError)."""
        return int(self._lib.mlc_hip_capture_end())

    def capturedLaunches(self, handle: int) -> int:
        return int(self._lib.mlc_hip_captured_launches(handle))

    def replayUpdate(self, handle, page_tables_flat, page_table_offsets, seq_lens, q_positions,
                     page_ids=None, slots_in_page=None) -> bool:
        return self._call.replay_update(handle, page_tables_flat, page_table_offsets, seq_lens, q_positions, page_ids,
                                        slots_in_page)

    def replay(self, handle: int) -> bool:
        return self._call.replay(handle)

    def captureRelease(self, handle: int) -> None:
        self._lib.mlc_hip_capture_release(handle)

    # -- measurement helpers
    def timerStart(self) -> bool:
        return bool(self._lib.mlc_hip_timer_start())

    def timerStopMs(self) -> float:
        return float(self._lib.mlc_hip_timer_stop())

    def lastDecodeLaunches(self) -> int:
        return int(self._lib.mlc_hip_last_decode_launches())

    def lastDecodeWorkItems(self) -> int:
        return int(self._lib.mlc_hip_last_decode_work_items())

    def lastDecodeKernel(self) -> str:
        return (self._lib.mlc_hip_last_decode_kernel() or b"").decode()

    def tableUploads(self) -> int:
        """Times so far the decode path copied a page table to the device."""
        return int(self._lib.mlc_hip_decode_table_uploads())

    def fusedKvWriteLaunches(self) -> int:
        """KV writes so far that went out fused with a neighbour (option "fuse_row_ops")."""
        return int(self._lib.mlc_hip_fused_kv_write_launches())

    def kvWritesInDecodeLaunches(self) -> int:
        """Decode attention launches so far that carried the step's KV write."""
        return int(self._lib.mlc_hip_kv_writes_in_decode_launches())

    def fusedMatmulRopeLaunches(self) -> int:
        """Q4_0 matmuls so far launched with the split + RoPE + cast of their output as epilogue."""
        return int(self._lib.mlc_hip_fused_matmul_rope_launches())

    def fusedMatmulSiluLaunches(self) -> int:
        """Q4_0 matmuls so far launched with the gate/up split + SiLU * up of their output as epilogue."""
        return int(self._lib.mlc_hip_fused_matmul_silu_launches())

    def fusedMatmulSiluSplitLaunches(self) -> int:
        """... of which also wrote the activation fragments of the matmul that reads the products."""
        return int(self._lib.mlc_hip_fused_matmul_silu_split_launches())

    def fusedDecodeSplitLaunches(self) -> int:
        """Decode attention launches so far that also wrote the next Q4_0 matmul's activation fragments."""
        return int(self._lib.mlc_hip_fused_decode_split_launches())

    def fusedMatmulNormLaunches(self) -> int:
        """Q4_0 matmuls so far launched with the residual add, the RMSNorm's sums and the next matmul's
        input as epilogue."""
        return int(self._lib.mlc_hip_fused_matmul_norm_launches())

    def rowProgramLaunches(self) -> int:
        """Held-back row operators so far that went out as one: chains, and adds behind a matmul (option "fuse_row_ops")."""
        return int(self._lib.mlc_hip_row_program_launches())

    def setOption(self, name: str, value: int) -> bool:
        return bool(self._lib.mlc_hip_set_option(name.encode(), int(value)))

    def stream(self) -> int:
        return self._lib.mlc_hip_stream() or 0
