"""CPU-side checks of the product library: it loads, exports every symbol the C
header declares, reads/validates `.ae8` packs with the reference's error
semantics, and its tokenizer reproduces the reference's id vectors."""
import json
import os
import re
import subprocess

import numpy as np
import pytest

import arctic_embed_amd as ae
from conftest import GOLDEN, ROOT

HEADER = os.path.join(ROOT, "include", "arctic_embed.h")


def declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(ae_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    names = declared_functions()
    assert len(names) >= 30
    out = subprocess.run(["nm", "-D", "--defined-only", ae.LIB_PATH], capture_output=True, text=True).stdout
    exported = set(re.findall(r" T (ae_[a-z0-9_]+)", out))
    missing = [n for n in names if n not in exported]
    assert not missing, missing
    for n in names:  # resolvable through the dynamic loader as well
        getattr(ae.lib(), n)


def test_noalloc_attention_refuses_before_any_device_work():
    """ae_attention_varlen_noalloc refuses sizes past its static scratch (524288 records: two plan
    lists of 4 + 12 (total_tokens / 32 + n_seqs + 1) records plus (n_seqs + 4) / 4 for the checked
    cu_seqlens) and a max_seq_len outside 1..512 from the arguments alone, before it touches a
    device pointer: no device addresses are passed here."""
    lib = ae.lib()
    call = lambda n, t, max_len: lib.ae_attention_varlen_noalloc(None, None, n, t, max_len, None, None)
    assert call(60000, 1 << 20, 512) == ae.AE_ERR_CAPACITY
    assert "static scratch" in lib.ae_last_error().decode()
    # the largest batch of one-token segments that fits: 2 (4 + 12 (n/32 + n + 1)) + (n + 4)/4 <= 524288
    fits = lambda n: 2 * (4 + 12 * (n // 32 + n + 1)) + (n + 4) // 4 <= 524288
    n_max = max(n for n in range(20000, 22000) if fits(n))
    assert call(n_max + 1, n_max + 1, 1) == ae.AE_ERR_CAPACITY
    assert call(n_max, n_max, 1) == ae.AE_ERR_INVALID_ARG  # fits: only then the null pointers are refused
    assert call(2, 100, 513) == ae.AE_ERR_INVALID_ARG
    assert call(2, 100, 0) == ae.AE_ERR_INVALID_ARG
    assert call(3, 2, 64) == ae.AE_ERR_INVALID_ARG  # fewer tokens than segments


@pytest.mark.parametrize("lens,choice", [
    # a workgroup per compute unit: single sequences up to 168 tokens, a few short ones
    ([65], 2), ([128], 2), ([129], 2), ([160], 2), ([168], 2), ([169], 1), ([509], 1),
    ([66, 66], 2), ([80, 80], 2), ([140, 16], 2), ([80, 20, 20, 20], 2), ([112, 20, 20], 2),
    ([128, 128], 1), ([88, 90], 1), ([100, 60, 20], 1), ([70] + [8] * 9, 1),
    ([64], 0), ([128] * 12, 0)])
def test_attention_choice(lens, choice):
    """Which kernels the exact attention takes by the batch (256 compute units)."""
    assert ae.attention_choice(len(lens), sum(lens), max(lens), max(lens)) == choice


@pytest.mark.parametrize("n_seqs,tokens,bound,longest,choice", [
    # 16-query tiles beyond 1,024 tokens: the longest row over 1.5 times the mean; as launched by
    # embed_batch (bound: the longest up to a power of two)
    (32, 8192, 512, 260, 0), (104, 7168, 128, 66, 0), (64, 8192, 256, 130, 0), (24, 7168, 512, 300, 0),
    # up to 16 segments, by the bound
    (12, 2843, 512, 506, 1), (16, 4040, 400, 398, 1), (16, 9001, 512, 512, 0), (8, 2048, 512, 260, 1),
    # more, with rows over 400 keys: further where the longest row is known
    (17, 4353, 502, 502, 1), (30, 8985, 496, 496, 1), (30, 9001, 496, 496, 0),
    (20, 2490, 512, 0, 1), (20, 2501, 512, 0, 0), (20, 5138, 512, 0, 0),
    # more, up to 400 keys: not unless the rows are mostly short
    (24, 1669, 127, 127, 0), (40, 6265, 260, 260, 0), (32, 7963, 385, 385, 0), (17, 4420, 400, 0, 0),
    (64, 1578, 100, 100, 1), (200, 4000, 100, 100, 1), (200, 4774, 100, 100, 0), (60, 1024, 512, 0, 1),
    # mostly short rows behind a long one, or behind a bound of 512
    (130, 3764, 512, 512, 1), (130, 5087, 512, 0, 1), (200, 9000, 512, 0, 1), (200, 9001, 512, 0, 0)])
def test_attention_choice_by_the_longest_row(n_seqs, tokens, bound, longest, choice):
    assert ae.attention_choice(n_seqs, tokens, bound, longest) == choice


@pytest.mark.parametrize("m,n,k,residual,rows16", [
    # K = 1024 and 1536 without a residual: 7 and 8 workgroups per compute unit (slower beyond: up to 1.42 times)
    (3584, 384, 1024, False, True), (3585, 384, 1024, False, False), (4096, 384, 1536, False, True),
    (4097, 384, 1536, False, False), (6144, 384, 1536, False, False), (2048, 768, 1024, False, False),
    (1184, 1152, 1024, False, True), (1536, 1152, 1024, False, False), (1040, 1536, 1024, False, False),
    # with one: 12
    (6144, 384, 1536, True, True), (6145, 384, 1536, True, False), (3072, 768, 1024, True, True),
    (6144, 384, 1024, True, True), (2048, 1152, 1024, True, True), (1537, 1536, 1536, True, False),
    # K = 384: one round, with or without
    (6144, 384, 384, False, True), (2048, 1152, 384, True, True), (2049, 1152, 384, True, False),
    # no K split
    (1025, 384, 768, False, False)])
def test_gemm_tile_height_rule(m, n, k, residual, rows16):
    """Which int8 GEMMs beyond 1,024 rows keep the 16-row workgroups (256 compute units): those for
    which these measured faster than the 64 x 192 tiles."""
    assert ae.gemm_int8_rows16(m, n, k, residual) == rows16


def test_version_and_default_dir(monkeypatch):
    assert "gfx950" in ae.version()
    monkeypatch.setenv("ARCTIC_EMBED_MODEL_DIR", "/some/dir")
    assert ae.default_model_dir() == "/some/dir"
    monkeypatch.delenv("ARCTIC_EMBED_MODEL_DIR")
    assert ae.default_model_dir() == "model"


def test_cosine_similarity():
    rng = np.random.default_rng(0)
    a = rng.normal(size=384).astype(np.float32)
    b = rng.normal(size=384).astype(np.float32)
    s = np.float32(0)
    for i in range(384):  # sequential f32 dot (src/lib.rs:265-271)
        s = np.float32(s + a[i] * b[i])
    assert ae.cosine_similarity(a, b) == s


def _open_code(ae8, vocab):
    try:
        e = ae.Engine.from_files(ae8, vocab)
    except ae.AeError as err:
        return err.code
    e.close()
    return ae.AE_OK


def test_pack_errors_follow_reference(tmp_path, model_dir):
    data = open(str(model_dir / "model.ae8"), "rb").read()
    vocab = str(model_dir / "vocab.txt")
    assert _open_code(str(tmp_path / "none.ae8"), vocab) == ae.AE_ERR_NOT_FOUND
    assert _open_code(str(model_dir / "model.ae8"), str(tmp_path / "none.txt")) == ae.AE_ERR_NOT_FOUND
    bad = tmp_path / "bad.ae8"
    bad.write_bytes(b"ARCTIC9\x01" + data[8:])
    assert _open_code(str(bad), vocab) == ae.AE_ERR_INVALID_DATA
    for cut in (3, 8, 100, len(data) - 10):
        t = tmp_path / ("t%d.ae8" % cut)
        t.write_bytes(data[:cut])
        assert _open_code(str(t), vocab) == ae.AE_ERR_EOF, cut


def test_valid_pack_without_gpu_reports_unsupported(model_dir):
    torch = pytest.importorskip("torch")
    if torch.cuda.is_available():
        pytest.skip("GPU present")
    assert _open_code(str(model_dir / "model.ae8"), str(model_dir / "vocab.txt")) == ae.AE_ERR_UNSUPPORTED


def test_tokenizer_reference_vectors():
    tok = ae.Tokenizer(os.path.join(GOLDEN, "vocab.txt"))
    assert tok.vocab_size() == 30522
    d = json.load(open(os.path.join(GOLDEN, "tokenizer_vectors.json"), encoding="utf-8"))
    assert len(d["short"]) == 12 and len(d["long"]) == 7
    for r in d["short"]:  # tests/accuracy_test.rs:86-96
        ids = tok.encode_query(r["raw_text"]) if r["kind"] == "query" else tok.encode(r["raw_text"])
        assert list(ids) == r["ids"], r["raw_text"]
    for r in d["long"]:  # examples/dump_ids.rs: BertTokenizer::encode per line
        assert list(tok.encode(r["text"])) == r["ids"], r["name"]


def test_tokenizer_edge_cases():
    tok = ae.Tokenizer(os.path.join(GOLDEN, "vocab.txt"))
    assert list(tok.encode("")) == [101, 102]
    assert list(tok.encode("\x00�\x07")) == [101, 102]     # removed by the normalizer
    assert list(tok.encode("HELLO")) == list(tok.encode("hello"))  # lowercase
    assert list(tok.encode("café")) == list(tok.encode("cafe"))  # accent stripping
    assert list(tok.encode("café")) == list(tok.encode("cafe"))  # combining mark dropped
    long = tok.encode("word " * 1000)
    assert len(long) == 512 and long[0] == 101 and long[-1] == 102
    q = tok.encode_query("x")
    assert len(q) > 3 and q[0] == 101 and q[-1] == 102
    assert list(tok.encode("a" * 101)) == [101, 100, 102]  # > 100 chars -> [UNK]
    assert list(tok.encode("中文"))[1:-1] == list(tok.encode("中 文"))[1:-1]


RUST_FFI = os.path.join(ROOT, "snowflake-arctic-embed-s-rust_amd", "rust", "src", "ffi.rs")
_C_TO_RUST = {"int": "c_int", "size_t": "usize", "uint16_t": "u16", "uint32_t": "u32", "uint64_t": "u64",
              "int8_t": "i8", "int32_t": "i32", "float": "f32", "double": "f64", "char": "c_char", "void": "c_void"}


def _rust_type_of_c(ctype):
    """A C type as the Rust FFI type that binds it: each pointer is *const when what it points
    to is const, else *mut; opaque ae_* structs keep their names."""
    toks = re.findall(r"const|\*|\w+", ctype)
    base = [t for t in toks if t not in ("const", "*")]
    assert len(base) == 1, ctype
    level_const, ptrs, seen_ptr = False, [], False
    for t in toks:
        if t == "const":
            level_const = True
        elif t == "*":
            ptrs.append("*const" if level_const else "*mut")
            level_const, seen_ptr = False, True
    name = _C_TO_RUST.get(base[0], base[0])
    if not ptrs and name == "c_void":
        return None
    return " ".join(list(reversed(ptrs)) + [name])


def _header_signatures():
    text = re.sub(r"/\*.*?\*/", "", open(HEADER).read(), flags=re.S)
    text = re.sub(r"^\s*#.*$", "", text, flags=re.M)
    sigs = {}
    for ret, name, args in re.findall(r"^[ \t]*([A-Za-z_][\w \t\*]*?)\b(ae_[a-z0-9_]+)\s*\(([^)]*)\)\s*;", text,
                                      flags=re.M):
        params = []
        for a in [a.strip() for a in args.split(",") if a.strip() and a.strip() != "void"]:
            ctype = re.sub(r"\b\w+$", "", a).strip()  # drop the parameter name
            params.append(_rust_type_of_c(ctype))
        sigs[name] = (_rust_type_of_c(ret.strip()), params)
    return sigs


def test_rust_binding_matches_the_header():
    """The Rust crate's raw declarations (snowflake-arctic-embed-s-rust_amd/rust/src/ffi.rs; no
    Rust toolchain in this image) bind each entry point with the header's parameter count and
    types, and cover every entry point other than the ae_debug_* test hooks."""
    sigs = _header_signatures()
    text = open(RUST_FFI).read()
    block = text[text.index('extern "C" {'):]
    rust = {}
    for name, args, ret in re.findall(r"pub fn (ae_[a-z0-9_]+)\(([^)]*)\)\s*(?:->\s*([^;]+?))?\s*;", block, flags=re.S):
        params = [" ".join(p.split(":", 1)[1].split()) for p in args.split(",") if p.strip()]
        rust[name] = (" ".join(ret.split()) if ret else None, params)
    assert rust, "no declarations parsed"
    for name, (ret, params) in rust.items():
        assert name in sigs, name
        assert (ret, params) == sigs[name], (name, (ret, params), sigs[name])
    missing = [n for n in sigs if n not in rust and not n.startswith("ae_debug_")]
    assert not missing, missing
    # the constants the crate mirrors
    for const in ("AE_OK", "AE_ERR_NOT_FOUND", "AE_ERR_INVALID_DATA", "AE_ERR_EOF", "AE_ERR_INVALID_ARG",
                  "AE_ERR_UNSUPPORTED", "AE_ERR_CAPACITY", "AE_ERR_HIP", "AE_ATTENTION_EXACT",
                  "AE_ATTENTION_QUANTIZED", "AE_KERNEL_KINDS", "AE_HIDDEN_SIZE"):
        cval = re.search(r"#define %s \(?(-?\d+)\)?" % const, open(HEADER).read()).group(1)
        rval = re.search(r"pub const %s: \w+ = (-?\d+);" % const, text).group(1)
        assert cval == rval, const
