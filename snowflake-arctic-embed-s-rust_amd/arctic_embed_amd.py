"""ctypes binding of libarctic_embed_amd.so (the C ABI in include/arctic_embed.h).

Python mirror of the reference API (mdlockyer/snowflake-arctic-embed-s-rust,
src/lib.rs): ``ArcticEmbedS.from_dir`` -> ``Engine.from_dir``, ``Workspace``,
``embed_tokens`` / ``embed_query`` / ``embed_document`` / ``embed_batch``, plus
the operator-level entry points.  The library is loaded from this directory;
there is no fallback: a missing library raises ``ImportError``.

Device pointers are plain integers (e.g. ``torch.Tensor.data_ptr()``).
"""
import ctypes
import os

import numpy as np

HIDDEN = 384
INTER = 1536
MAX_POS = 512
VOCAB = 30522

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libarctic_embed_amd.so")

if not os.path.exists(LIB_PATH):
    raise ImportError(
        "libarctic_embed_amd.so is not built (run __graft_entry__.build() or make -C %s)" % _HERE)

# One process must hold one HIP runtime.  PyTorch-ROCm ships its own
# libamdhip64 (SONAME libamdhip64.so.7) and asks for it as "libamdhip64.so";
# this library asks for "libamdhip64.so.7".  Loading torch first lets our
# dependency resolve to torch's copy by SONAME; loading ours first would make
# torch map a second runtime, and the two then fight over the device.
try:
    import torch  # noqa: F401
except ImportError:
    pass
_lib = ctypes.CDLL(LIB_PATH)

_c = ctypes
_vp, _sz, _i32, _u64, _f32p = _c.c_void_p, _c.c_size_t, _c.c_int, _c.c_uint64, _c.POINTER(_c.c_float)

_SIGS = {
    "ae_last_error": (_c.c_char_p, []),
    "ae_version": (_c.c_char_p, []),
    "ae_engine_open": (_i32, [_c.c_char_p, _c.POINTER(_vp)]),
    "ae_engine_open_files": (_i32, [_c.c_char_p, _c.c_char_p, _c.POINTER(_vp)]),
    "ae_engine_close": (None, [_vp]),
    "ae_engine_size_bytes": (_sz, [_vp]),
    "ae_engine_raw_size_bytes": (_sz, [_vp]),
    "ae_default_model_dir": (_sz, [_c.c_char_p, _sz]),
    "ae_workspace_create": (_i32, [_vp, _sz, _sz, _c.POINTER(_vp)]),
    "ae_workspace_destroy": (None, [_vp]),
    "ae_workspace_stream": (_vp, [_vp]),
    "ae_embed_tokens": (_i32, [_vp, _vp, _vp, _sz, _vp]),
    "ae_embed_query": (_i32, [_vp, _vp, _c.c_char_p, _vp]),
    "ae_embed_document": (_i32, [_vp, _vp, _c.c_char_p, _vp]),
    "ae_embed_batch": (_i32, [_vp, _vp, _c.POINTER(_c.c_char_p), _sz, _i32, _i32, _vp]),
    "ae_embed_batch_tokens": (_i32, [_vp, _vp, _vp, _vp, _sz, _vp]),
    "ae_forward_packed_device": (_i32, [_vp, _vp, _vp, _vp, _i32, _i32, _i32, _vp, _vp]),
    "ae_cosine_similarity": (_c.c_float, [_vp, _vp]),
    "ae_linear_create": (_i32, [_i32, _i32, _vp, _vp, _vp, _vp, _c.POINTER(_vp)]),
    "ae_linear_destroy": (None, [_vp]),
    "ae_gemm_w8a8": (_i32, [_vp, _i32, _vp, _vp, _vp, _vp, _vp]),
    "ae_layernorm_smooth_quantize": (_i32, [_i32, _vp, _vp, _vp, _vp, _vp, _vp, _vp]),
    "ae_smooth_quantize": (_i32, [_i32, _i32, _vp, _vp, _vp, _vp, _vp]),
    "ae_gelu_smooth_quantize": (_i32, [_i32, _i32, _vp, _vp, _vp, _vp, _vp]),
    "ae_attention_varlen": (_i32, [_vp, _vp, _i32, _i32, _vp, _vp]),
    "ae_attention_varlen_quantized": (_i32, [_vp, _vp, _i32, _i32, _vp, _vp]),
    "ae_workspace_attention_varlen": (_i32, [_vp, _vp, _vp, _i32, _i32, _i32, _vp, _vp]),
    "ae_workspace_attention_varlen_quantized": (_i32, [_vp, _vp, _vp, _i32, _i32, _i32, _vp, _vp]),
    "ae_workspace_synchronize": (_i32, [_vp, _vp]),
    "ae_attention_varlen_noalloc": (_i32, [_vp, _vp, _i32, _i32, _i32, _vp, _vp]),
    "ae_write_synthetic_ae8": (_i32, [_c.c_char_p, _u64]),
    "ae_tokenizer_open": (_i32, [_c.c_char_p, _c.POINTER(_vp)]),
    "ae_tokenizer_close": (None, [_vp]),
    "ae_tokenizer_encode": (_i32, [_vp, _c.c_char_p, _i32, _vp, _sz, _c.POINTER(_sz)]),
    "ae_tokenizer_vocab_size": (_sz, [_vp]),
    "ae_debug_gelu_map": (_i32, [_vp, _vp, _sz, _vp]),
    "ae_debug_mfma_products": (_i32, [_vp, _vp, _vp, ctypes.c_int, _vp]),
    "ae_debug_set_attention_form": (_i32, [ctypes.c_int]),
    "ae_debug_attention_choice": (_i32, [ctypes.c_int] * 5),
    "ae_debug_gemm_int8_rows16": (_i32, [ctypes.c_int] * 5),
    "ae_debug_set_ffn_rows": (_i32, [ctypes.c_int]),
    "ae_debug_set_ffn_exact_gelu": (_i32, [ctypes.c_int]),
    "ae_debug_gelu_fast_certify": (_i32, [ctypes.POINTER(ctypes.c_uint64)]),
    "ae_debug_ffn_repairs": (_i32, [ctypes.POINTER(ctypes.c_uint64), ctypes.POINTER(ctypes.c_uint64), ctypes.c_int]),
    "ae_workspace_set_timing": (_i32, [_vp, _i32]),
    "ae_workspace_set_graphs": (_i32, [_vp, _i32]),
    "ae_workspace_set_attention_mode": (_i32, [_vp, _i32]),
    "ae_debug_forward_prefix": (_i32, [_vp, _vp, _vp, _vp, _sz, _i32, _vp, _vp, _vp]),
    "ae_workspace_kernel_times": (_i32, [_vp, _vp, _vp]),
    "ae_debug_gemm_quant_a": (_i32, [_vp, _i32, _vp, _vp, _vp, _vp, _vp, _vp]),
    "ae_debug_gemm_gelu": (_i32, [_vp, _i32, _vp, _vp, _vp, _vp, _vp, _vp]),
    "ae_debug_gemm_ln": (_i32, [_vp, _i32, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp]),
    "ae_debug_ffn": (_i32, [_vp, _vp, _i32, _vp, _vp, _vp, _vp, _vp]),
    "ae_debug_ffn_ln": (_i32, [_vp, _vp, _i32] + [_vp] * 11),
    "ae_parallel_context_create": (_i32, [_vp, _i32, _c.POINTER(_vp)]),
    "ae_parallel_context_destroy": (None, [_vp]),
    "ae_parallel_context_threads": (_i32, [_vp]),
    "ae_embed_tokens_parallel": (_i32, [_vp, _vp, _vp, _sz, _vp]),
    "ae_embed_query_parallel": (_i32, [_vp, _vp, _c.c_char_p, _vp]),
    "ae_embed_document_parallel": (_i32, [_vp, _vp, _c.c_char_p, _vp]),
}
for _name, (_res, _args) in _SIGS.items():
    _fn = getattr(_lib, _name)
    _fn.restype = _res
    _fn.argtypes = _args

# status codes (include/arctic_embed.h)
AE_OK, AE_ERR_NOT_FOUND, AE_ERR_INVALID_DATA, AE_ERR_EOF = 0, -1, -2, -3
AE_ERR_INVALID_ARG, AE_ERR_UNSUPPORTED, AE_ERR_CAPACITY, AE_ERR_HIP = -4, -5, -6, -7


KERNEL_KINDS = ("embed_ln", "gemm_qkv", "attention", "gemm_attn_out", "ln1", "gemm_ffn_up", "gemm_ffn_down", "ln2",
                "layer11_tail")


class AeError(RuntimeError):
    def __init__(self, code, msg):
        super().__init__("ae error %d: %s" % (code, msg))
        self.code = code


def lib():
    return _lib


def _check(rc):
    if rc != AE_OK:
        raise AeError(rc, (_lib.ae_last_error() or b"").decode(errors="replace"))


def version():
    return _lib.ae_version().decode()


def write_synthetic_ae8(path, seed):
    """Seeded synthetic model in .ae8 layout."""
    _check(_lib.ae_write_synthetic_ae8(str(path).encode(), int(seed)))


def default_model_dir():
    n = _lib.ae_default_model_dir(None, 0)
    buf = ctypes.create_string_buffer(n)
    _lib.ae_default_model_dir(buf, n)
    return buf.value.decode()


def cosine_similarity(a, b):
    a = np.ascontiguousarray(a, dtype=np.float32)
    b = np.ascontiguousarray(b, dtype=np.float32)
    return float(_lib.ae_cosine_similarity(a.ctypes.data, b.ctypes.data))


def _wsh(ws):
    """A workspace's handle, or None: the engine's own workspace (grown on demand)."""
    return ws.handle if ws is not None else None


def _pack_ids(seqs):
    lens = [len(s) for s in seqs]
    offsets = np.zeros(len(seqs) + 1, dtype=np.uint32)
    offsets[1:] = np.cumsum(lens)
    ids = np.concatenate([np.asarray(s, dtype=np.uint16) for s in seqs]) if seqs else np.zeros(0, np.uint16)
    return np.ascontiguousarray(ids, dtype=np.uint16), offsets


class Tokenizer:
    """BertTokenizer (src/tokenizer.rs:26-208)."""

    def __init__(self, vocab_path):
        h = ctypes.c_void_p()
        _check(_lib.ae_tokenizer_open(str(vocab_path).encode(), ctypes.byref(h)))
        self._h = h

    def vocab_size(self):
        return int(_lib.ae_tokenizer_vocab_size(self._h))

    def _enc(self, text, is_query):
        buf = np.zeros(MAX_POS, dtype=np.uint16)
        n = ctypes.c_size_t()
        _check(_lib.ae_tokenizer_encode(self._h, text.encode("utf-8"), 1 if is_query else 0, buf.ctypes.data,
                                        buf.size, ctypes.byref(n)))
        return buf[:n.value].copy()

    def encode(self, text):
        return self._enc(text, False)

    def encode_query(self, text):
        return self._enc(text, True)

    def close(self):
        if self._h:
            _lib.ae_tokenizer_close(self._h)
            self._h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


class Engine:
    """ArcticEmbedS (src/lib.rs:34-72): device-resident weights, shared by threads."""

    def __init__(self, handle):
        self._h = handle

    @classmethod
    def from_dir(cls, path=None):
        h = ctypes.c_void_p()
        _check(_lib.ae_engine_open(None if path is None else str(path).encode(), ctypes.byref(h)))
        return cls(h)

    @classmethod
    def from_files(cls, ae8_path, vocab_path=None):
        h = ctypes.c_void_p()
        _check(_lib.ae_engine_open_files(str(ae8_path).encode(),
                                         None if vocab_path is None else str(vocab_path).encode(),
                                         ctypes.byref(h)))
        return cls(h)

    @property
    def handle(self):
        return self._h

    def size_bytes(self):
        return int(_lib.ae_engine_size_bytes(self._h))

    def raw_size_bytes(self):
        return int(_lib.ae_engine_raw_size_bytes(self._h))

    def close(self):
        if self._h:
            _lib.ae_engine_close(self._h)
            self._h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def workspace(self, max_tokens=0, max_seqs=0):
        return Workspace(self, max_tokens, max_seqs)

    # --- embedding API (src/lib.rs:76-260) ---
    def embed_tokens(self, ws, ids):
        ids = np.ascontiguousarray(ids, dtype=np.uint16)
        out = np.zeros(HIDDEN, dtype=np.float32)
        _check(_lib.ae_embed_tokens(self._h, _wsh(ws), ids.ctypes.data, ids.size, out.ctypes.data))
        return out

    def embed_batch_tokens(self, ws, seqs):
        ids, offsets = _pack_ids(list(seqs))
        out = np.zeros((len(offsets) - 1, HIDDEN), dtype=np.float32)
        _check(_lib.ae_embed_batch_tokens(self._h, _wsh(ws), ids.ctypes.data, offsets.ctypes.data,
                                          len(offsets) - 1, out.ctypes.data))
        return out

    def embed_query(self, ws, text):
        out = np.zeros(HIDDEN, dtype=np.float32)
        _check(_lib.ae_embed_query(self._h, _wsh(ws), text.encode("utf-8"), out.ctypes.data))
        return out

    def embed_document(self, ws, text):
        out = np.zeros(HIDDEN, dtype=np.float32)
        _check(_lib.ae_embed_document(self._h, _wsh(ws), text.encode("utf-8"), out.ctypes.data))
        return out

    def embed_batch(self, ws, texts, is_query=False, num_threads=1):
        n = len(texts)
        arr = (ctypes.c_char_p * max(n, 1))(*[t.encode("utf-8") for t in texts])
        out = np.zeros((n, HIDDEN), dtype=np.float32)
        _check(_lib.ae_embed_batch(self._h, _wsh(ws), arr, n, 1 if is_query else 0, int(num_threads),
                                   out.ctypes.data))
        return out

    # --- latency mode (src/lib.rs:104-133) ---
    def parallel_context(self, n_threads):
        return ParallelContext(self, n_threads)

    def embed_tokens_parallel(self, ids, par):
        ids = np.ascontiguousarray(ids, dtype=np.uint16)
        out = np.zeros(HIDDEN, dtype=np.float32)
        _check(_lib.ae_embed_tokens_parallel(self._h, par.handle, ids.ctypes.data, ids.size, out.ctypes.data))
        return out

    def embed_query_parallel(self, text, par):
        out = np.zeros(HIDDEN, dtype=np.float32)
        _check(_lib.ae_embed_query_parallel(self._h, par.handle, text.encode("utf-8"), out.ctypes.data))
        return out

    def embed_document_parallel(self, text, par):
        out = np.zeros(HIDDEN, dtype=np.float32)
        _check(_lib.ae_embed_document_parallel(self._h, par.handle, text.encode("utf-8"), out.ctypes.data))
        return out

    def forward_prefix(self, ws, seqs, layers):
        """Embedding + `layers` encoder layers; returns (hidden, act_q, act_scale) over packed rows."""
        ids, offsets = _pack_ids(list(seqs))
        T = int(offsets[-1])
        hidden = np.zeros((T, HIDDEN), np.float32)
        act_q = np.zeros((T, HIDDEN), np.int8)
        scale = np.zeros(T, np.float32)
        _check(_lib.ae_debug_forward_prefix(self._h, _wsh(ws), ids.ctypes.data, offsets.ctypes.data, len(offsets) - 1,
                                            int(layers), hidden.ctypes.data, act_q.ctypes.data, scale.ctypes.data))
        return hidden, act_q, scale

    def forward_packed_device(self, ws, ids_ptr, cu_ptr, n_seqs, total_tokens, out_ptr, stream=None,
                              max_seq_len=0):
        """forward_ragged_cls over a packed batch already in HBM (max_seq_len 0 = 512)."""
        _check(_lib.ae_forward_packed_device(self._h, _wsh(ws), ids_ptr, cu_ptr, int(n_seqs),
                                             int(total_tokens), int(max_seq_len), out_ptr, stream))


class Workspace:
    """Workspace (src/model.rs:123-173): HIP stream + device activations; one per thread."""

    def __init__(self, engine, max_tokens=0, max_seqs=0):
        h = ctypes.c_void_p()
        _check(_lib.ae_workspace_create(engine.handle, int(max_tokens), int(max_seqs), ctypes.byref(h)))
        self._h = h
        self._engine = engine

    @property
    def handle(self):
        return self._h

    @property
    def stream(self):
        return _lib.ae_workspace_stream(self._h)

    def set_timing(self, enabled):
        _check(_lib.ae_workspace_set_timing(self._h, 1 if enabled else 0))

    def set_graphs(self, enabled):
        """Graph replay of repeated forward passes (on by default); False forces eager launches."""
        _check(_lib.ae_workspace_set_graphs(self._h, 1 if enabled else 0))

    def set_attention_mode(self, quantized):
        """Layers 0-10 with the reference's ArmSme quantized attention (True) or the exact path."""
        _check(_lib.ae_workspace_set_attention_mode(self._h, 1 if quantized else 0))

    def synchronize(self, stream=None):
        """Waits for the workspace's work and raises AeError (AE_ERR_INVALID_ARG) if a device-resident
        batch since the last call failed its checks."""
        _check(_lib.ae_workspace_synchronize(self._h, stream))

    def attention_varlen(self, qkv_ptr, cu_ptr, n_seqs, total_tokens, max_seq_len, ctx_ptr, stream=None,
                         quantized=False):
        """ae_attention_varlen(_quantized) on this workspace's scratch: asynchronous, no allocation."""
        fn = _lib.ae_workspace_attention_varlen_quantized if quantized else _lib.ae_workspace_attention_varlen
        _check(fn(self._h, qkv_ptr, cu_ptr, int(n_seqs), int(total_tokens), int(max_seq_len), ctx_ptr, stream))

    def kernel_times(self):
        """{kind: (total_ms, launches)} since timing was enabled (synchronize first)."""
        ms = np.zeros(len(KERNEL_KINDS), np.float64)
        cnt = np.zeros(len(KERNEL_KINDS), np.int32)
        _check(_lib.ae_workspace_kernel_times(self._h, ms.ctypes.data, cnt.ctypes.data))
        return {k: (float(ms[i]), int(cnt[i])) for i, k in enumerate(KERNEL_KINDS)}

    def close(self):
        if self._h:
            _lib.ae_workspace_destroy(self._h)
            self._h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


class ParallelContext:
    """ParallelContext (src/parallel.rs:137-253): latency mode for one sequence at a time."""

    def __init__(self, engine, n_threads):
        h = ctypes.c_void_p()
        _check(_lib.ae_parallel_context_create(engine.handle, int(n_threads), ctypes.byref(h)))
        self._h = h

    @property
    def handle(self):
        return self._h

    @property
    def threads(self):
        return int(_lib.ae_parallel_context_threads(self._h))

    def close(self):
        if self._h:
            _lib.ae_parallel_context_destroy(self._h)
            self._h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


class Linear:
    """PackedLinearInt8 (src/gemm.rs:165-247) on the device."""

    def __init__(self, w_q, w_scale, bias, inv_smooth):
        w_q = np.ascontiguousarray(w_q, dtype=np.int8)
        self.n_out, self.k_in = w_q.shape
        self._keep = [np.ascontiguousarray(x, dtype=np.float32) for x in (w_scale, bias, inv_smooth)]
        h = ctypes.c_void_p()
        _check(_lib.ae_linear_create(self.n_out, self.k_in, w_q.ctypes.data, self._keep[0].ctypes.data,
                                     self._keep[1].ctypes.data, self._keep[2].ctypes.data, ctypes.byref(h)))
        self._h = h

    def gemm(self, m, a_ptr, a_scale_ptr, res_ptr, out_ptr, stream=None):
        """gemm_int8_fused (src/gemm.rs:630-671) on device pointers."""
        _check(_lib.ae_gemm_w8a8(self._h, int(m), a_ptr, a_scale_ptr, res_ptr, out_ptr, stream))

    def gemm_quant_a(self, m, x_ptr, rowmax_ptr, smooth_ptr, res_ptr, out_ptr, stream=None):
        """GEMM with A quantized on load from f32 rows (the attn_out / FFN-down variant)."""
        _check(_lib.ae_debug_gemm_quant_a(self._h, int(m), x_ptr, rowmax_ptr, smooth_ptr, res_ptr, out_ptr, stream))

    def gemm_ln(self, m, x_ptr, rowmax_ptr, smooth_ptr, res_ptr, gamma_ptr, beta_ptr, ln_smooth_ptr, dst_ptr, q_ptr,
                scale_ptr, stream=None):
        """The attention output GEMM (A quantized on load, smoothed, residual) and the LayerNorm +
        SmoothQuant of its rows in one kernel; its f32 output is not stored."""
        _check(_lib.ae_debug_gemm_ln(self._h, int(m), x_ptr, rowmax_ptr, smooth_ptr, res_ptr, gamma_ptr, beta_ptr,
                                     ln_smooth_ptr, dst_ptr, q_ptr, scale_ptr, stream))

    def gemm_gelu(self, m, a_ptr, a_scale_ptr, g_smooth_ptr, out_ptr, rowmax_ptr, stream=None):
        """GEMM with the GELU * smooth epilogue and row absmax (the FFN-up variant)."""
        _check(_lib.ae_debug_gemm_gelu(self._h, int(m), a_ptr, a_scale_ptr, g_smooth_ptr, out_ptr, rowmax_ptr, stream))

    def ffn(self, down, m, a_ptr, a_scale_ptr, res_ptr, out_ptr, stream=None):
        """The fused FFN block (src/model.rs:725-755) with this linear as FFN-up
        (384 -> 1536) and `down` as FFN-down (1536 -> 384); out may equal res."""
        _check(_lib.ae_debug_ffn(self._h, down._h, int(m), a_ptr, a_scale_ptr, res_ptr, out_ptr, stream))

    def ffn_ln(self, down, m, a_ptr, a_scale_ptr, res_ptr, out_ptr, gamma_ptr, beta_ptr, ln_smooth_ptr, dst_ptr, q_ptr,
               scale_ptr, stream=None):
        """ffn and the LayerNorm + SmoothQuant of its rows in one kernel (up to one round of 16-row
        workgroups)."""
        _check(_lib.ae_debug_ffn_ln(self._h, down._h, int(m), a_ptr, a_scale_ptr, res_ptr, out_ptr, gamma_ptr, beta_ptr,
                                    ln_smooth_ptr, dst_ptr, q_ptr, scale_ptr, stream))

    def close(self):
        if self._h:
            _lib.ae_linear_destroy(self._h)
            self._h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


def layernorm_smooth_quantize(m, x_ptr, gamma_ptr, beta_ptr, smooth_ptr, q_ptr, scale_ptr, stream=None):
    _check(_lib.ae_layernorm_smooth_quantize(int(m), x_ptr, gamma_ptr, beta_ptr, smooth_ptr, q_ptr, scale_ptr,
                                             stream))


def smooth_quantize(m, n, x_ptr, smooth_ptr, q_ptr, scale_ptr, stream=None):
    _check(_lib.ae_smooth_quantize(int(m), int(n), x_ptr, smooth_ptr, q_ptr, scale_ptr, stream))


def gelu_smooth_quantize(m, n, x_ptr, smooth_ptr, q_ptr, scale_ptr, stream=None):
    _check(_lib.ae_gelu_smooth_quantize(int(m), int(n), x_ptr, smooth_ptr, q_ptr, scale_ptr, stream))


def attention_varlen(qkv_ptr, cu_ptr, n_seqs, total_tokens, ctx_ptr, stream=None):
    _check(_lib.ae_attention_varlen(qkv_ptr, cu_ptr, int(n_seqs), int(total_tokens), ctx_ptr, stream))


def attention_varlen_noalloc(qkv_ptr, cu_ptr, n_seqs, total_tokens, max_seq_len, ctx_ptr, stream=None):
    """attention_varlen with no allocation, host copy or synchronization (static device scratch)."""
    _check(_lib.ae_attention_varlen_noalloc(qkv_ptr, cu_ptr, int(n_seqs), int(total_tokens), int(max_seq_len),
                                            ctx_ptr, stream))


def attention_varlen_quantized(qkv_ptr, cu_ptr, n_seqs, total_tokens, ctx_ptr, stream=None):
    """attention_varlen as the reference's ArmSme backend computes it (int8 Q/K/V, int16 P)."""
    _check(_lib.ae_attention_varlen_quantized(qkv_ptr, cu_ptr, int(n_seqs), int(total_tokens), ctx_ptr, stream))


def gelu_map(x_ptr, y_ptr, n, stream=None):
    _check(_lib.ae_debug_gelu_map(x_ptr, y_ptr, int(n), stream))


def mfma_products(a_ptr, b_ptr, out_ptr, n_sets, stream=None):
    """Raw results of the attention kernels' exact-product MFMA (16 floats per lane per set of 64 pairs)."""
    _check(_lib.ae_debug_mfma_products(a_ptr, b_ptr, out_ptr, int(n_sets), stream))


def set_attention_form(form):
    """Exact-attention kernels to launch from now on: 0 by the batch (default),
    1 tiled / register rows only, 2 the latency form only (a test hook)."""
    _check(_lib.ae_debug_set_attention_form(int(form)))


def attention_choice(n_seqs, total_tokens, max_seq_len, longest=0, cus=256):
    """The exact attention's kernels for a batch (longest: its longest row, 0 if only the bound
    max_seq_len is known): 0 tiles of 32 queries, 1 of 16, 2 the smallest batches' kernel (a test
    hook, no device access)."""
    return _lib.ae_debug_attention_choice(int(n_seqs), int(total_tokens), int(max_seq_len), int(longest), int(cus))


def gemm_int8_rows16(m, n, k, residual, cus=256):
    """Whether Linear.gemm of m > 1024 rows takes its 16-row workgroups on a GPU of cus compute
    units (a test hook, no device access)."""
    return bool(_lib.ae_debug_gemm_int8_rows16(int(m), int(n), int(k), 1 if residual else 0, int(cus)))


def set_ffn_rows(rows):
    """Token rows per workgroup of the fused FFN kernel from now on: 0 by the
    batch (default), 16, 32 or 64, or -m: the first m rows (a multiple of 64) in 64-row
    workgroups, the rest in 32-row ones (a test hook)."""
    _check(_lib.ae_debug_set_ffn_rows(int(rows)))


def set_ffn_exact_gelu(exact):
    """The fused FFN kernel's GELU from now on: False (default) the fast GELU with exact repair,
    True the reference's GELU on every element (a test hook; both give the same bits)."""
    _check(_lib.ae_debug_set_ffn_exact_gelu(1 if exact else 0))


def gelu_fast_certify():
    """The six counters of the exhaustive fast-GELU certification (ae_debug_gelu_fast_certify)."""
    out = (ctypes.c_uint64 * 6)()
    _check(_lib.ae_debug_gelu_fast_certify(out))
    return [int(x) for x in out]


def ffn_repairs(reset=False):
    """(tiles, rows): the fast FFN kernel's exact recomputations on the current device since the
    last reset: 16 x 16 tiles recomputed for an undecided quantized value, and the 16-row groups of
    the passes with more candidates for the row maxima than rows (a test hook)."""
    t, r = ctypes.c_uint64(0), ctypes.c_uint64(0)
    _check(_lib.ae_debug_ffn_repairs(ctypes.byref(t), ctypes.byref(r), 1 if reset else 0))
    return int(t.value), int(r.value)
