"""CPU-only checks: the C ABI library loads and exports every symbol the header declares,
the parameter blocks have the reference's layout, arguments are rejected with clear errors,
and the host-side mirror of the reference's types behaves as the reference's do.  Nothing
here computes on a GPU; on a box without one the library must refuse to run, loudly."""
import ctypes
import os
import re
import subprocess
import timeit

import pytest

import __graft_entry__ as entry

saetta = entry.load_package()
ffi = saetta.ffi
ROOT = entry.ROOT


def header_functions():
    text = open(os.path.join(ROOT, "include", "saetta_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(saetta_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    assert os.path.exists(ffi.LIB_PATH), "build the library first: python __graft_entry__.py"
    declared = header_functions()
    assert declared == sorted(ffi.SYMBOLS)
    out = subprocess.run(["nm", "-D", "--defined-only", ffi.LIB_PATH], capture_output=True, text=True, check=True).stdout
    exported = set(re.findall(r" T (saetta_[a-z0-9_]+)", out))
    assert set(declared) <= exported
    lib = ctypes.CDLL(ffi.LIB_PATH)
    for name in declared:
        assert hasattr(lib, name)


def test_header_is_plain_c():
    # The boundary is a C ABI: the header must compile as C99 on its own (a Rust, Go or C binding reads it).
    header = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include", "saetta_hip.h")
    done = subprocess.run(["gcc", "-std=c99", "-Wall", "-Wextra", "-pedantic", "-Werror", "-fsyntax-only", "-x", "c", header],
                          capture_output=True, text=True)
    assert done.returncode == 0, done.stderr
    # ... and the parameter blocks the mirrors build by hand have the sizes the compiler gives them
    probe = ('#include "%s"\n#include <stdio.h>\nint main(void) { printf("%%zu %%zu %%zu %%zu %%zu\\n", '
             'sizeof(saetta_rows_fused_params), sizeof(saetta_rows_step_params), sizeof(saetta_conv_rows_params), '
             'sizeof(saetta_step_params), sizeof(saetta_conv_params)); return 0; }\n') % header
    import tempfile
    with tempfile.TemporaryDirectory() as d:
        src, exe = os.path.join(d, "probe.c"), os.path.join(d, "probe")
        with open(src, "w") as f:
            f.write(probe)
        subprocess.run(["gcc", "-std=c99", src, "-o", exe], check=True)
        sizes = [int(x) for x in subprocess.run([exe], capture_output=True, text=True, check=True).stdout.split()]
    assert sizes == [ctypes.sizeof(ffi.RowsFusedParamsC), ctypes.sizeof(ffi.RowsStepParamsC), ctypes.sizeof(ffi.ConvRowsParamsC),
                     ctypes.sizeof(ffi.StepParamsC), ctypes.sizeof(ffi.ConvParamsC)]


def test_parameter_blocks_match_the_reference_layout():
    # TokenParams (src/plan.rs:16-35) is 4 x u32; DecodeParams 3 x u32 + f32 (src/attention.rs:19-26);
    # RowsAttentionParams adds rows, splits (src/rows.rs:307-317); FlashParams 4 x u32 + f32
    # (src/attention_prefill.rs:4-14); KvQuantParams 2 x u32 (src/kv_quant.rs:147-153).
    assert ctypes.sizeof(ffi.TokenParamsC) == 16
    assert ctypes.sizeof(ffi.DecodeParamsC) == 16 and ffi.DecodeParamsC.scale.offset == 12
    assert ctypes.sizeof(ffi.RowsParamsC) == 24 and ffi.RowsParamsC.rows.offset == 16
    assert ctypes.sizeof(ffi.FlashParamsC) == 20 and ffi.FlashParamsC.scale.offset == 16
    assert ctypes.sizeof(ffi.KvQuantParamsC) == 8
    assert ctypes.sizeof(ffi.QuantRowsC) == 24


def test_scratch_sizes_never_exceed_the_reference():
    lib = ffi.lib()
    for capacity in (1, 100, 128, 1024, 32896, 150016, 262144):
        chunks = -(-capacity // 128)
        for rows in (1, 4, 8):
            assert lib.saetta_part_o_bytes(16, capacity, rows) <= rows * chunks * 16 * 256 * 4
            assert lib.saetta_part_ml_bytes(16, capacity, rows) <= rows * chunks * 16 * 2 * 4
            assert lib.saetta_part_o_bytes(16, capacity, rows) == 128 * lib.saetta_part_ml_bytes(16, capacity, rows)


def test_bad_arguments_are_rejected_before_any_launch():
    lib = ffi.lib()
    rows = ffi.QuantRowsC(16, 16, 16)
    p = ffi.KvQuantParamsC(8, 8)
    assert lib.saetta_kv_quantize(None, 5, 16, rows, p, None, 0) == -1  # SAETTA_E_BITS
    assert b"bits 5" in lib.saetta_last_error()
    assert lib.saetta_kv_quantize(None, 8, None, rows, p, None, 0) == -3  # SAETTA_E_NULL
    assert lib.saetta_kv_quantize(None, 8, 12, rows, p, None, 0) == -4  # x not 16-byte aligned
    dp = ffi.DecodeParamsC(16, 4, 1024, 0.0625)
    assert lib.saetta_attn_decode_quant(None, 8, 16, rows, rows, 16, 16, 16, 16, dp, 16, 3) == -2
    assert b"8 q heads per kv head" in lib.saetta_last_error()
    rp = ffi.RowsParamsC(16, 2, 1024, 0.0625, 9, 8)
    assert lib.saetta_attn_rows_quant(None, 8, 16, rows, rows, 16, 16, 16, 16, rp, 16, 3) == -2
    assert b"9 rows" in lib.saetta_last_error()
    odd = ffi.DecodeParamsC(16, 2, 1000, 0.0625)
    assert lib.saetta_attn_decode_quant(None, 8, 16, rows, rows, 16, 16, 16, 16, odd, 16, 3) == -2
    assert b"multiple of 16" in lib.saetta_last_error()
    # Gated DeltaNet: heads must divide, v_dim a multiple of 4 for several tokens, snapshots need a buffer
    sp = ffi.RowsStepParamsC(2, 3, 8, 1, 1e-6, 0)
    assert lib.saetta_deltanet_rows(None, *([16] * 9), None, sp) == -2
    assert b"value heads" in lib.saetta_last_error()
    sp = ffi.RowsStepParamsC(1, 2, 6, 1, 1e-6, 0)
    assert lib.saetta_deltanet_rows(None, *([16] * 9), None, sp) == -2
    sp = ffi.RowsStepParamsC(1, 2, 8, 1, 1e-6, 1)
    assert lib.saetta_deltanet_rows(None, *([16] * 9), None, sp) == -3  # snapshots asked for, no buffer
    cp = ffi.ConvRowsParamsC(64, 1, 4, 0)
    assert lib.saetta_deltanet_conv_rows(None, 16, 16, 16, 16, None, cp) == -2
    assert b"kernel size" in lib.saetta_last_error()
    # ... the fused call takes up to 8 rows, conv kernels of 2..16 taps, and both snapshot buffers or neither
    fused = ffi.RowsFusedParamsC(1, 2, 8, 4, 1e-6, 9, 0)
    assert lib.saetta_deltanet_rows_fused(None, *([16] * 11), None, None, fused) == -2
    assert b"9 rows" in lib.saetta_last_error()
    fused = ffi.RowsFusedParamsC(1, 2, 8, 17, 1e-6, 2, 0)
    assert lib.saetta_deltanet_rows_fused(None, *([16] * 11), None, None, fused) == -2
    assert b"kernel size" in lib.saetta_last_error()
    fused = ffi.RowsFusedParamsC(1, 2, 8, 4, 1e-6, 2, 1)
    assert lib.saetta_deltanet_rows_fused(None, *([16] * 11), 16, None, fused) == -3
    fused = ffi.RowsFusedParamsC(1, 2, 8, 4, 1e-6, 2, 0)
    assert lib.saetta_deltanet_rows_fused(None, *([16] * 7), 12, *([16] * 3), None, None, fused) == -4  # the state's alignment
    token_c, token_s = ffi.ConvParamsC(100, 4), ffi.StepParamsC(1, 2, 8, 1e-6)
    assert lib.saetta_deltanet_token(None, *([16] * 11), token_c, token_s) == -2
    assert b"channels" in lib.saetta_last_error()
    fp = ffi.FlashParamsC(16, 2, 0, 1, 0.0625)
    assert lib.saetta_attn_prefill_quant(None, 16, 16, rows, rows, 16, 16, fp, None, 0) == -1
    assert lib.saetta_attn_prefill_quant(None, 8, 16, rows, rows, 16, 16, fp, 8, 1 << 30) == -4  # workspace alignment
    # 32 keys per image, one image per kv head and block, whole kilobytes each; behind them a 256-byte line
    # (the attention kernel's count of tiles handed out)
    one = lib.saetta_prefill_workspace_bytes(0, 32, 1) - 256
    assert one % 1024 == 0 and one >= 2 * 32 * 256 * 2
    assert lib.saetta_prefill_workspace_bytes(4096, 4096, 2) == one * 2 * 256 + 256
    assert lib.saetta_prefill_workspace_bytes(0, 33, 1) == 2 * one + 256
    with pytest.raises(ffi.SaettaError):
        ffi.check(-1, "demo")


def test_without_a_gpu_the_library_refuses_to_run():
    import torch
    if torch.cuda.is_available():
        pytest.skip("this box has a GPU")
    rc = ffi.lib().saetta_init()
    assert rc == -5  # SAETTA_E_DEVICE: there is no CPU fallback
    assert ffi.lib().saetta_last_error()


def test_calls_check_what_they_are_given():
    import torch
    # what the extension refuses before it asks for a stream: types, layouts, sizes, each copy of the package with its own error
    x, h, ap, p = torch.zeros(512), torch.zeros(512, dtype=torch.float16), saetta.attention_prefill, saetta.FlashParams(16, 2, 0, 1, 0.0625)
    for bad in (x, x.numpy(), None, "x"):
        with pytest.raises(TypeError, match=r"to_half x: expected a contiguous torch.float32 tensor on the GPU"):
            saetta.to_half(bad, h)
    rows = saetta.QuantRows(saetta.KvBits.Eight, 512, 4, "cpu")
    with pytest.raises(TypeError, match="QuantRows.encode x"):
        rows.encode(x, 0, 1)
    for pos, tokens in ((-1, 1), (-4, 8), (0, -1), (3, -1), (4, 1), (0, 5), (2**63 - 1, 1), (-2**63, 0)):
        with pytest.raises(ValueError, match="tokens do not fit"):
            rows.encode(x, pos, tokens)
    with pytest.raises(ValueError, match="no prefill attention kernel"):
        ap.encode("attention_fa3", h, h, h, x, x, p, workspace=x)
    with pytest.raises(ValueError, match="attention_fa4 needs 8 q heads per kv head"):
        ap.encode("attention_fa4", h, h, h, x, x, saetta.FlashParams(15, 2, 0, 1, 0.0625), workspace=x)
    with pytest.raises(ValueError, match="attention_fa4 needs 8 q heads per kv head"):  # ... before there is a workspace
        ap.encode("attention_fa4", h, h, h, x, x, saetta.FlashParams(15, 2, 0, 1, 0.0625))
    with pytest.raises(ValueError, match="prefill attention needs 8 q heads per kv head"):
        ap.encode_quant(h, rows, rows, x, x, saetta.FlashParams(15, 2, 0, 1, 0.0625))
    with pytest.raises(TypeError, match="q: expected a contiguous torch.float16"):
        ap.encode("attention_fa8", h, h, h, x, x, p, workspace=x)
    calls = saetta.host._calls
    with pytest.raises(TypeError, match="token_params_set params: expected a tensor on the GPU"):
        calls.token_params_set(x, 0, 0, 0, 0)
    with pytest.raises(TypeError, match="expected FlashParams"):
        calls.prefill("attention_fa8", h, h, h, x, x, "p", x, None)
    with pytest.raises(TypeError, match="takes 3 arguments"):
        calls.to_half(x, h)
    with pytest.raises(saetta.ffi.SaettaError, match="plan_run: .*code"):
        calls.plan_run(0, 0)


def test_the_calls_extension_is_looked_for_when_it_is_called(tmp_path):
    # loaded by the import where it is there; a package imported before its extension is there: importing works, a call says
    # what is missing, and works once it is built; one that does not load is an error of the call, too
    assert "to_half" in vars(ffi.calls)
    import shutil
    import sys
    src = os.path.dirname(ffi.__file__)
    shutil.copytree(src, tmp_path / "pkg", ignore=shutil.ignore_patterns("*.so", "*.o", "__pycache__", "csrc"))
    os.makedirs(tmp_path / "pkg" / "lib", exist_ok=True)
    code = f"""
import os, shutil, torch, pkg
x = torch.zeros(64)
def raised():
    try:
        pkg.to_half(x, x)
    except Exception as e:
        return e
e = raised()
assert isinstance(e, pkg.ffi.SaettaError) and "is missing" in str(e), e
with open(pkg.ffi.CALLS_PATH, "w") as f:
    f.write("not a library")
e = raised()
assert isinstance(e, pkg.ffi.SaettaError) and "does not load" in str(e), e
os.remove(pkg.ffi.CALLS_PATH)
shutil.copy({ffi.CALLS_PATH!r}, pkg.ffi.CALLS_PATH)
e = raised()
assert type(e) is TypeError and "to_half x" in str(e), e
"""
    subprocess.run([sys.executable, "-c", code], check=True, cwd=tmp_path, env=dict(os.environ, PYTHONPATH=str(tmp_path)))


def test_the_library_is_built_without_torch(tmp_path):
    # what make would do: with a Python that finds no torch, or none at all, the C library and nothing else; the extension by the
    # Python that is asked for, under the name which that Python looks for
    import sys

    def steps(python, *goals):
        r = subprocess.run(["make", "-n", "-B", "-C", os.path.join(ROOT, "saetta-macqwen_amd", "csrc"), f"PYTHON={python}", *goals], capture_output=True, text=True)
        return r.returncode, r.stdout + r.stderr

    bare = tmp_path / "bare"
    bare.write_text(f'#!/bin/sh\nexec {sys.executable} -S -I "$@"\n')  # (without site-packages)
    bare.chmod(0o755)
    for python in (bare, tmp_path / "none"):
        rc, text = steps(python)
        assert rc == 0 and "libsaetta_hip.so" in text and "calls" not in text, text
        rc, text = steps(python, "calls")
        assert rc != 0 and "need torch" in text
    rc, text = steps(sys.executable)
    assert rc == 0 and os.path.basename(ffi.CALLS_PATH) in text and "libsaetta_hip.so" in text


def test_the_extension_is_this_pythons(monkeypatch):
    # built by the Python that runs build(), whatever python3 is on the path, and under a name that no other loads
    import sys
    import sysconfig
    made = []
    monkeypatch.setattr(entry.subprocess, "run", lambda command, **_: made.append(command))
    entry.build()
    assert f"PYTHON={sys.executable}" in made[0] and "calls" in made[0]
    assert ffi.CALLS_PATH.endswith("_saetta_calls" + sysconfig.get_config_var("EXT_SUFFIX"))


def test_kv_bits_mirror():
    # src/kv_quant.rs:11-50
    K = saetta.KvBits
    assert K.parse("16") is K.Half and K.parse("8") is K.Eight and K.parse("4") is K.Four and K.parse("2") is None
    assert [k.bits() for k in (K.Half, K.Eight, K.Four)] == [16, 8, 4]
    assert K.Eight.words_per_group() == 16 and K.Four.words_per_group() == 8
    assert K.Half.bytes_per_value() == 2.0
    assert K.Eight.bytes_per_value() == 1.0 + 4.0 / 64 and K.Four.bytes_per_value() == 0.5 + 4.0 / 64
    # bytes per token and kv head of 256: 272 at 8 bits, 144 at 4 (src/kv_quant.rs:3-4)
    assert K.Eight.bytes_per_value() * 256 == 272 and K.Four.bytes_per_value() * 256 == 144
    assert saetta.GROUP == 64 and saetta.MAX_ROWS == 8


def test_token_params_and_prefill_constants():
    tp = saetta.TokenParams(7, 41)
    assert (tp.token, tp.position, tp.kv_len, tp.pad) == (7, 41, 42, 0)  # src/plan.rs:26-34
    ap = saetta.attention_prefill
    assert ap.KERNELS == ["attention_fa8", "attention_fa4"] and ap.DEFAULT == "attention_fa8" and ap.KEY_BLOCK == 16
    p = saetta.FlashParams(16, 2, 5, 8, 0.0625).c()
    assert (p.heads, p.kv_heads, p.pos, p.tokens) == (16, 2, 5, 8)


def test_plan_records_and_filters_ops_without_a_device():
    plan = saetta.Plan.__new__(saetta.Plan)  # no device buffer: only the op list is exercised
    plan.ops = []
    ran = []
    plan.op("attention_partial_mma_q8", lambda s: ran.append("partial"))
    plan.op("attention_reduce", lambda s: ran.append("reduce"))
    built = plan.build_where(lambda name: name == "attention_reduce")
    assert [k for k, _ in built.ops] == ["attention_reduce"]
    assert [k for k, _ in plan.build().ops] == ["attention_partial_mma_q8", "attention_reduce"]


@pytest.mark.parametrize("pos,tokens,kv,parts", [(4096, 4096, 2, 0), (2048, 2048, 2, 0), (300, 16, 1, 3), (20000, 4096, 2, 2), (118784, 2048, 2, 2),
                                                 (60007, 1237, 2, 3), (3000, 2300, 2, 4), (86225, 447, 2, 7), (10000, 100, 2, 12), (20000, 12, 2, 32)])
def test_parts_of_a_chunks_keys(pos, tokens, kv, parts):
    # what the layouts' estimates come to on 256 CUs: whole keys, wide tiles in 2 to 7 parts, tiles of 16 in 3 to 32
    images = -(-(pos + tokens) // 32) * kv * 32768 + 256
    assert ffi.lib().saetta_prefill_workspace_bytes(pos, tokens, kv) - images == parts * -(-tokens // 16) * kv * 16 * 8 * (1024 + 8)


def test_the_plan_of_a_long_chunk_costs_the_host_no_more_than_a_short_ones():
    # every call makes one: few layouts of many rounds are worked out to their end
    size = ffi.lib().saetta_prefill_workspace_bytes
    of = lambda *chunk: min(timeit.repeat(lambda: size(*chunk), number=500, repeat=20))  # noqa: E731
    assert of(20000, 4096, 2) < 2 * of(20000, 12, 2)


def test_the_librarys_own_workspace_takes_less_where_there_is_less(tmp_path):
    # (its memory comes from a function of the caller's: here one that has a limit and counts)
    src, exe = tmp_path / "take.cc", tmp_path / "take"
    src.write_text("""
#include "owned_workspace.hpp"
#include <cstdio>
static size_t limit = SIZE_MAX, held = 0;
static int asked = 0, given_back = 0;
static char memory[1];
int main() {
    saetta::OwnedWorkspace w;
    auto take = [&](std::initializer_list<size_t> wants) {
        asked = given_back = 0;
        const bool ok = w.take(wants, [](size_t n) -> void * { asked++; return held || n > limit ? nullptr : (held = n, memory); },
                               [](void *) { given_back++; held = 0; });
        printf("%d %zu %d %d\\n", ok, w.bytes, asked, given_back);
        if (ok != (w.ptr != nullptr) || held != w.bytes) puts("wrong");
    };
    take({100, 50, 40});   // the first
    take({90, 50, 40});    // is there
    limit = 120;
    take({200, 120, 110}); // refused: the second
    take({200, 120, 110}); // not asked for again
    take({300, 200, 110}); // nor is more
    limit = 130;
    take({200, 130});      // the last is more than is held
    take({150, 140});      // not even the last: nothing is held
    take({150, 60});       // 60 of it
    limit = 1000;
    take({150, 145});      // what was refused may be there by now, where nothing else does
    take({500, 400});      // and then anything is asked for
    take({500, 0});
}
""")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "saetta-macqwen_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    said = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split("\n")[:-1]
    assert said == ["1 100 1 0", "1 100 0 0", "1 120 2 1", "1 120 0 0", "1 120 0 0", "1 130 1 1", "0 0 2 1", "1 60 1 0", "1 145 1 1", "1 500 1 1", "1 500 0 0"]


def test_asm_that_changes_scc_says_so(tmp_path):
    # Most scalar arithmetic writes SCC, where the compiler may keep a comparison across a statement that does not name it.
    writes = re.compile(r"\bs_(add|sub|min|max|and|or|xor|not|andn2|orn2|nand|nor|xnor|lshl|lshr|ashr|bfe|bcnt|abs|cmp|bitcmp|wqm|quadmask|ff0|flbit|addk|cmpk)[a-z0-9]*_")
    folder, seen = os.path.join(ROOT, "saetta-macqwen_amd", "csrc"), 0
    for name in sorted(n for n in os.listdir(folder) if n.endswith((".hip", ".hpp"))):
        with open(os.path.join(folder, name)) as f:
            text = re.sub(r"(?m)^\s*#\s*(include|pragma).*$", "", f.read())  # (asm text is made of a file's own macros)
        text = subprocess.run(["g++", "-E", "-P", "-x", "c++", "-"], input=text, capture_output=True, text=True, check=True).stdout
        for at in re.finditer(r"\basm\b\s*(volatile\b\s*)?\(", text):
            statement = text[at.end():text.index(");", at.end())]
            seen += 1
            assert not writes.search(statement) or '"scc"' in statement, f"{name}: {statement}"
    assert seen > 50
