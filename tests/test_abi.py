"""The C-ABI library loads and exports every symbol include/zipage_hip.h declares.
No compute calls: this runs without a GPU."""
import ctypes
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared(header="zipage_hip.h"):
    text = open(os.path.join(ROOT, "include", header)).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(zp_[a-z_0-9]+)\s*\(", text)))


def test_header_declares_expected_entry_points():
    names = _declared()
    for n in ["zp_store_query", "zp_attention_score", "zp_global_score", "zp_pool_scores",
              "zp_key_norm", "zp_redundancy_lightning", "zp_redundancy_raw", "zp_score_epilogue",
              "zp_topk_mask", "zp_compress_kv", "zp_compress_score", "zp_last_error",
              "zp_abi_version"]:
        assert n in names


def test_library_exports_every_declared_symbol():
    from zipage_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.fail(f"{_lib.LIB_PATH} not built (python -m zipage_amd.build)")
    lib = ctypes.CDLL(_lib.LIB_PATH)
    for name in _declared():
        assert hasattr(lib, name), f"{name} declared in the header but not exported"
    assert sorted(_lib.EXPORTS) == _declared()


def test_models_library_exports_every_declared_symbol():
    from zipage_amd import _lib
    names = _declared("zipage_models.h")
    assert sorted(n for names in _lib.MODEL_EXPORTS.values() for n in names) == names
    for part, exported in _lib.MODEL_EXPORTS.items():
        lib = _lib.load_models(part)
        for name in exported:
            assert hasattr(lib, name), f"{name} declared in the header but not exported"
    lib = _lib.load_models("latent")
    # bad arguments are refused on the host, before any launch
    assert lib.zp_headwise_linear(None, None, None, None, None, 1, 2, 33, 16, 0, 0, 0, None) != 0
    assert b"multiples of 32" in lib.zp_last_error()
    assert lib.zp_latent_rows_attention(None, None, None, None, None, None, 1, 1, 32, 0, 16, 1, 1, 1, -1, 1.0, 0,
                                        None, 0, None) == 1
    lib = _lib.load_models("models")
    assert lib.zp_embed_norm(None, None, None, None, None, None, None, None, None, None, 1, 12, 12, 5, 5, 1.0, 1e-6, 0.0, 0.0, 0, None) != 0
    assert lib.zp_run_attention(None, None, None, None, None, None, None, None, 1, 4, 3, 32, 0, 32, 0, 0, 1, 1, 128, 256, 0,
                                128, 1.0, 1.0, 0, None) == 1
    lib = _lib.load_models("grouped")
    two = _lib.AttentionForm(0.0, 2, 0.5, 1e-6, 0, None, 0)                              # a mean over nothing
    assert lib.zp_grouped_rows_attention(1, 1, 1, 1, 1, None, ctypes.byref(two), 1, 1, 2, 2, 32, 32, 16, 1, 1, 1, 0, 0,
                                         64, 1.0, 1.0, 0, None, 0, None) == 1
    assert b"mean over the values" in lib.zp_last_error()
    lib = _lib.load_models("moe")
    assert lib.zp_moe_select(None, None, None, None, 1, 12, 5, 3, 1, 0, 12, None) == 1      # five of a group of four
    assert lib.zp_small_linear(None, None, None, 1, 40, 4, 40, 0, None) != 0
    lib = _lib.load_models("recurrent")
    bad = _lib.MlstmArgs(heads=2, dk=48, dv=32, vdim=32, cap=1.0, gate_stride=4, out_stride=64,
                         seg=_lib.Segments(n=1, num_slots=1, num_rows=1))
    assert lib.zp_mlstm_scan(ctypes.byref(bad), 0, None) != 0 and b"48" in lib.zp_last_error()
    bad = _lib.DeltaArgs(heads=3, kv_heads=2, dk=32, dv=32, vdim=32, taps=4, out_stride=96,
                         seg=_lib.Segments(n=1, num_slots=1, num_rows=1))
    assert lib.zp_delta_scan(ctypes.byref(bad), 0, None) == 1
    lib = _lib.load_models("linear")
    bad = _lib.LinearArgs(heads=2, dk=48, dv=32, vdim=32, in_stride=512, out_stride=64, seg=_lib.Segments(n=1, num_slots=1, num_rows=1))
    assert lib.zp_linear_scan(ctypes.byref(bad), 0, None) != 0 and b"48" in lib.zp_last_error()
    bad.dk, bad.rot = 32, 34                                                             # more than a head has
    assert lib.zp_linear_runs(ctypes.byref(bad), 0, 16, None, 0, 0, None) == 1


def test_version_and_error_string():
    from zipage_amd import _lib
    lib = _lib.load()
    assert lib.zp_abi_version() >= 2
    assert isinstance(lib.zp_last_error(), bytes)


def test_argument_validation_needs_no_gpu():
    """Bad arguments are rejected on the host before any launch."""
    from zipage_amd import _lib
    lib = _lib.load()
    rc = lib.zp_topk_mask(None, None, 4, 16, 17, 0, None)
    assert rc == 1 and b"k=17" in lib.zp_last_error()
    rc = lib.zp_global_score(1, 1, 1, 1, 1, 1, 1, 256, 8, 4, 0, 0, 1.5, 0, 1, 0, None)
    assert rc == 1 and b"decay_factor" in lib.zp_last_error()


def test_product_has_no_cpu_fallback():
    import torch
    from zipage_amd.kernel import topk_mask
    with pytest.raises(RuntimeError, match="device tensors"):
        topk_mask(torch.zeros(2, 8), 3)


def test_a_workspace_for_the_largest_batch_serves_every_other():
    from zipage_amd import _lib
    from zipage_amd.compress import CompressConfig, c_config
    lib = _lib.load()
    for kw in (dict(), dict(use_redudancy=True, use_global_score=True, decay_factor=0.8)):
        cc = c_config(CompressConfig(budget_blocks=8, query_cache_len=16, **kw))
        for dtype, heads, window in ((0, 32, 32), (1, 16, 16), (2, 16, 32)):
            sizes = [lib.zp_compress_layers_workspace(1, b, 9, 256, 8, heads, window, dtype, ctypes.byref(cc), 0) for b in range(1, 70)]
            assert sizes == sorted(sizes)
            few = [lib.zp_compress_layers_workspace_few(1, b, 9, 256, 8, heads, window, dtype, ctypes.byref(cc), 0) for b in range(1, 70)]
            assert few[0] > sizes[0] and few[-1] == sizes[-1] and all(f >= s for f, s in zip(few, sizes))


def test_room_for_halves_of_blocks_only_where_they_are_used():
    """Blocks of rows go in halves where the selection adds them up: not in the scorer's own call, nor for maxima over the window, nor where
    carried scores are looked at in between."""
    from zipage_amd import _lib
    from zipage_amd.compress import CompressConfig, c_config
    lib = _lib.load()
    size = lambda name, batch, cc=(), heads=32, dtype=0: getattr(lib, name)(1, batch, 9, 256, 8, heads, 32, dtype, *cc)
    for batch in (3, 4):                                                     # 96 and 128 blocks, too many for tiles
        assert size("zp_attention_score_workspace_few", batch) == size("zp_attention_score_workspace_for", batch)
    room = {}
    for name, kw in (("sums", {}), ("max", dict(reduced="max")), ("carried", dict(use_global_score=True, decay_factor=0.8)),
                     ("max norm", dict(use_global_score=True, decay_factor=0.8, max_norm=True)),
                     ("atomic", dict(use_global_score=True, decay_factor=0.8))):
        config = c_config(CompressConfig(budget_blocks=8, query_cache_len=32, **kw))
        config.deterministic_carry = name != "atomic"
        cc = (ctypes.byref(config), 0)
        for batch in (4, 5):
            room[name, batch] = size("zp_compress_layers_workspace_few", batch, cc) - size("zp_compress_layers_workspace", batch, cc)
    partials = 4 * 9 * 256 * 8 * 4 * 4                                       # of 128 blocks
    assert {k: v for k, v in room.items() if v} == {("sums", 4): 3 * partials, ("carried", 4): 3 * partials}


def test_room_for_few_sequences_fits_the_librarys_scratch():
    from zipage_amd import _lib
    from zipage_amd.compress import CompressConfig, c_config
    lib = _lib.load()
    header = open(os.path.join(ROOT, "include", "zipage_hip.h")).read()
    most = int(re.search(r"ZP_STATIC_SCRATCH_BYTES \((\d+)u << 20\)", header).group(1)) << 20
    for kw in (dict(), dict(use_redudancy=True, use_global_score=True, decay_factor=0.8), dict(reduced="max")):
        cc = (ctypes.byref(c_config(CompressConfig(budget_blocks=1, query_cache_len=16, **kw))), 1)
        for dtype in (0, 2):
            for NB, BS in ((40, 64), (20, 128), (10, 256), (1, 2560)):           # 2560 tokens
                for group in (1, 2, 4, 8):
                    for rows in range(1, 130):
                        size = [getattr(lib, "zp_compress_layers_workspace" + few)(1, rows, NB, BS, 1, group, 16, dtype, *cc) for few in ("_few", "")]
                        assert size[0] == size[1] or size[0] <= most


@pytest.mark.parametrize("NB,BS", [(52, 256), (26, 512), (202, 64), (1, 13120)])
def test_rows_beyond_the_limit_of_all_pairs_are_refused(NB, BS):
    from zipage_amd import _lib
    lib, p = _lib.load(), ctypes.c_void_p(4096)
    for dtype in (0, 1):
        size = lib.zp_redundancy_raw_workspace(1, 1, NB, BS, 1)
        assert lib.zp_redundancy_raw(p, p, p, None, 1, 1, NB, BS, 1, 128, NB, NB * BS * 128, BS * 128, 0.5, 0.4, dtype, p, size, None) == 3
        assert b"at most 13120 tokens and pages" in lib.zp_last_error()


def test_room_for_pieces_of_runs_follows_the_rows():
    """Blocks of 16 tokens alone where no run can be cut, as many states as rows, runs and heads can ask for beyond, and never more
    than 384."""
    from zipage_amd import _lib
    recurrent, linear = _lib.load_models("recurrent"), _lib.load_models("linear")
    for size, state in ((lambda *a: recurrent.zp_delta_runs_workspace(*a, 128, 128), 2 * 128 * 128 * 4),
                        (lambda *a: linear.zp_linear_runs_workspace(*a, 128), (128 * 128 + 128) * 4),
                        (lambda *a: recurrent.zp_mlstm_runs_workspace(*a), (128 * 128 + 128 + 4) * 4)):
        blocks = lambda rows, runs, heads: size(rows, runs, 1000) // 1000 * heads        # so many heads' runs stay whole
        for heads in (1, 8, 32, 128):
            assert size(16, 1, heads) == blocks(16, 1, heads) and size(192, 1, heads) == blocks(192, 1, heads)
        for rows, runs, heads in ((700, 1, 16), (1025, 3, 2), (2048, 1, 32), (16384, 8, 16)):
            room = size(rows, runs, heads) - blocks(rows, runs, heads)
            assert room == min(384, (rows // 64 + runs) * heads) * state
        assert size(2048, 8, 32) == blocks(2048, 8, 32)                                   # 256 pairs


def test_version_is_the_headers():
    from zipage_amd import _lib
    text = open(os.path.join(ROOT, "include", "zipage_hip.h")).read()
    assert _lib.ABI_VERSION == int(re.search(r"#define ZP_ABI_VERSION (\d+)", text)[1])
    for lib in (_lib.load(), *(_lib.load_models(name) for name in _lib.MODEL_LIBS)):
        assert lib.zp_abi_version() == _lib.ABI_VERSION


def test_library_of_another_version_is_refused(tmp_path):
    from zipage_amd import _lib
    path = str(tmp_path / "old.so")
    source = f"int zp_abi_version(void) {{ return {_lib.ABI_VERSION - 1}; }}"
    subprocess.run(["gcc", "-shared", "-fPIC", "-x", "c", "-", "-o", path], input=source, text=True, check=True)
    with pytest.raises(RuntimeError, match=f"ABI version {_lib.ABI_VERSION - 1}"):
        _lib._open(path, {}, {})


def test_structures_are_as_long_as_the_headers(tmp_path):
    from zipage_amd import _lib
    here = {"zp_compress_config": _lib.CompressConfigC, "zp_branch": _lib.Branch, "zp_segments": _lib.Segments, "zp_mlstm": _lib.MlstmArgs,
            "zp_delta": _lib.DeltaArgs, "zp_linear": _lib.LinearArgs, "zp_attention_form": _lib.AttentionForm, "zp_store_form": _lib.StoreForm}
    headers = "".join(open(os.path.join(ROOT, "include", h)).read() for h in ("zipage_hip.h", "zipage_models.h"))
    records = [n for n in re.findall(r"^} (zp_\w+);", headers, re.M)]
    assert sorted(records) == sorted(here)
    # the last field of each too: what lies behind the others has their sizes and places
    last = lambda t: t._fields_[-1][0]
    body = "".join(f'printf("%zu %zu\\n", sizeof({n}), offsetof({n}, {last(here[n])}));' for n in records)
    source = f'#include <stddef.h>\n#include <stdio.h>\n#include "zipage_hip.h"\n#include "zipage_models.h"\nint main(void) {{ {body} return 0; }}'
    exe = str(tmp_path / "sizes")
    subprocess.run(["gcc", "-I", os.path.join(ROOT, "include"), "-x", "c", "-", "-o", exe], input=source, text=True, check=True)
    out = subprocess.run([exe], capture_output=True, text=True, check=True).stdout.split("\n")
    for n, line in zip(records, out):
        assert [int(v) for v in line.split()] == [ctypes.sizeof(here[n]), getattr(here[n], last(here[n])).offset], n


def test_delta_products_of_other_ranks_are_refused():
    from zipage_amd import _lib
    lib = _lib.load_models("recurrent")
    args = _lib.DeltaArgs(in_stride=4096)
    call = lambda at, a_rank, rank: lib.zp_delta_runs_projected(ctypes.byref(args), ctypes.c_void_p(16), at, a_rank, rank, 0, 16, None, 0, 0, None)
    for at, a_rank, rank in ((4, 8, 16), (8, 8, 20), (0, 136, 144), (0, 16, 144), (0, 128, 264)):
        assert call(at, a_rank, rank) == 3, (at, a_rank, rank)             # ZP_EUNSUPPORTED
    assert call(4000, 64, 128) == 1 and call(0, 16, 8) == 1 and call(-8, 8, 16) == 1
