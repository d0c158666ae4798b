"""How the engine library comes by the kernel library: beside itself, where it is told, or from the program that loaded
it (the Python package compiles the kernels at the first call that needs them).  Runs without a GPU: the engine asks the
kernel library for its limits when it checks a configuration."""
import ctypes
import json
import os
import re
import shutil
import subprocess

import pytest

import test_gpu_kernels
from tq_kv_amd import kernels, native
from tq_kv_amd.csrc import build

CONFIG = {"architectures": ["Qwen2ForCausalLM"], "model_type": "qwen2", "hidden_size": 64, "num_hidden_layers": 1, "num_attention_heads": 2,
          "num_key_value_heads": 1, "intermediate_size": 96, "vocab_size": 50, "max_position_embeddings": 64, "rms_norm_eps": 1e-6,
          "rope_theta": 10000.0, "tie_word_embeddings": True}


def lonely_engine(tmp_path):
    """A copy of the engine library in a folder that holds no kernel library, loaded as a library of its own."""
    copy = os.path.join(str(tmp_path), "libtqengine_copy.so")
    shutil.copy(native.library_path(), copy)
    lib = ctypes.CDLL(copy)
    lib.tqe_write_random_folder.restype = ctypes.c_int
    lib.tqe_write_random_folder.argtypes = [ctypes.c_char_p, ctypes.c_char_p, ctypes.c_uint64, ctypes.c_int]
    lib.tqe_last_error.restype = ctypes.c_char_p
    lib.tqe_kernel_library.restype = ctypes.c_char_p
    return lib


def test_the_engine_asks_its_loader_for_the_kernels_when_it_finds_none(tmp_path, monkeypatch):
    monkeypatch.delenv("TQ_KERNEL_LIBRARY", raising=False)
    lib = lonely_engine(tmp_path)
    text = json.dumps(CONFIG).encode()

    def write(name):             # builds the model's parts, which ask the kernels what sizes they take
        return lib.tqe_write_random_folder(os.path.join(str(tmp_path), name).encode(), text, 1, native.BF16)
    assert write("a") == native.ERR_DEVICE
    assert b"kernel library is not built" in lib.tqe_last_error()
    # a builder that cannot: the same error
    kind = ctypes.CFUNCTYPE(ctypes.c_void_p)
    calls = []
    cannot = kind(lambda: calls.append("cannot"))
    lib.tqe_set_kernel_builder.argtypes = [kind]
    lib.tqe_set_kernel_builder.restype = None
    lib.tqe_set_kernel_builder(cannot)
    assert write("b") == native.ERR_DEVICE and calls == ["cannot"]
    # one that can is asked once, and the library it names is the one in use from then on
    path = ctypes.create_string_buffer(kernels.library_path().encode())

    def build():
        calls.append("can")
        return ctypes.addressof(path)
    can = kind(build)
    lib.tqe_set_kernel_builder(can)
    assert write("c") == 0, lib.tqe_last_error()
    assert sorted(os.listdir(os.path.join(str(tmp_path), "c"))) == ["config.json", "model.safetensors"]
    assert write("d") == 0 and calls == ["cannot", "can"]
    assert lib.tqe_kernel_library() == path.value


def test_the_float32_product_of_few_rows_issues_its_loads_in_the_stages_order(tmp_path):
    """Its waits let the 24 youngest loads be under way, which are the three later stages' only while every stage's eight loads are issued
    together, in the stages' order, from the first one on: read off the compiled kernel."""
    asm = os.path.join(str(tmp_path), "gemm_generic.s")
    subprocess.run([build._hipcc()] + build.HIPCC_FLAGS + ["-I", build.HERE, "--offload-device-only", "-S", os.path.join(build.HERE, "gemm_generic.hip"), "-o", asm],
                   check=True, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    with open(asm) as f:
        body = re.search(r"^_Z20gemm_few_rows_kernel\w+:[^\n]*\n(.*?)^\.Lfunc_end", f.read(), re.S | re.M).group(1)
    kinds = {"buffer_load_dwordx4": "w", "global_load_dwordx4": "x"}
    events = []
    for line in body.splitlines():
        word = line.split()[:2]
        if word and word[0] in kinds:
            events.append(kinds[word[0]])
        elif word and word[0] == "s_waitcnt" and "vmcnt" in line:
            events.append(word[1])
    stage = ["w"] * 4 + ["x"] * 4
    # three stages ahead, then four turns of a stage's loads and the wait for the one three before it, then the wait for all
    assert events[:3 * 8 + 4 * 9 + 1] == stage * 3 + (stage + ["vmcnt(24)"]) * 4 + ["vmcnt(0)"]


def test_the_sizes_of_the_prompt_products_tests_take_every_tile():
    """The choice is made on the host: every tile of the table is taken by some size, the ones without a gate both with K whole and (where real
    sizes do that) in pieces."""
    lib = kernels.library()
    whole = {kernels.prompt_tile(*size) for size in test_gpu_kernels.PROMPT_SIZES if lib.tqk_prompt_splits(*size) == 1}
    cut = [kernels.prompt_tile(*size) for size in test_gpu_kernels.PROMPT_SIZES if lib.tqk_prompt_splits(*size) > 1]
    gated = {kernels.prompt_tile(m, 2 * inter, k, True) for m, inter, k in test_gpu_kernels.PROMPT_GATED_SIZES}
    assert whole == set(range(9)) and len(cut) == 7 and set(cut) >= {1, 3, 4, 5, 6, 8}
    assert gated == {0, 1, 4, 5, 6, 7, 8, 9}            # three tiles a wave have no gate and up side by side; the last is the gate's alone
    assert kernels.prompt_tile(129, 16, 250) == -1


def test_the_sizes_of_the_mid_products_tests_take_every_tile():
    """Tiles a wave takes, by the rows' groups (up to 32, 64 and 128 rows); gated products always take pairs."""
    taken = {}
    for m, n, k in test_gpu_kernels.MID_LONG_SIZES:
        assert kernels.library().tqk_mid_splits(n, k, 0) == 1
        taken.setdefault(32 if m <= 32 else 64 if m <= 64 else 128, set()).add(kernels.mid_tile(m, n, k)[0])
    assert taken == {32: {1, 2, 5}, 64: {1, 2, 6}, 128: {1, 2, 3}}
    assert kernels.mid_tile(64, 2 * 8960, 1536, True) == (2, 3)


@pytest.mark.parametrize("m,n,k,gated,pays", [
    (200, 512, 4096, False, False), (129, 128, 2048, False, False), (8000, 32, 1024, False, False), (1024, 16, 512, False, False),  # small and cut
    (2048, 512, 256, False, True), (300, 512, 256, False, True),                                                                  # not cut
    (129, 3584, 18944, False, True), (300, 3584, 18944, False, True), (232, 1536, 8960, False, True),                             # cut and large
    (200, 128, 8192, True, False), (129, 2048, 8192, True, False), (512, 1024, 4096, True, False),                                # long K, few blocks
    (129, 37888, 3584, True, True), (255, 37888, 3584, True, True), (1023, 17920, 1536, True, True), (768, 55296, 5120, True, True),
    (129, 37888, 3584 + 32, True, False), (129, 24, 256, False, False)])                                                           # not taken at all
def test_which_products_pay_in_the_kernel_for_prompts(m, n, k, gated, pays):
    assert kernels.prompt_pays(m, n, k, gated) == pays


def small_step(**sizes):
    """What the kernel for small models' steps is asked about: a TqkSmallStep, its pointers left out."""
    class Layer(ctypes.Structure):
        _fields_ = [("pointers", ctypes.c_void_p * 9), ("eps1", ctypes.c_float), ("eps2", ctypes.c_float), ("scale", ctypes.c_float),
                    ("window", ctypes.c_int), ("table", ctypes.c_int), ("width", ctypes.c_int), ("divided", ctypes.c_int)]

    class Step(ctypes.Structure):
        _fields_ = [("pointers", ctypes.c_void_p * 7), ("final_eps", ctypes.c_float)] + [(n, ctypes.c_int) for n in (
            "act_dtype max_positions n_layers hidden n_heads n_kv_heads head_dim inter vocab n_rows n_want n_ints tokens tok_seq tok_pos want seq_first last_rows "
            "n_seqs decode max_end n_last").split()] + [("layers", Layer * 16), ("ints", ctypes.c_int32 * 400)]
    return Step(**dict(dict(act_dtype=1, max_positions=128, n_layers=2, hidden=64, n_heads=4, n_kv_heads=2, head_dim=16, inter=160, vocab=256, n_rows=1, n_want=1,
                            n_seqs=1, decode=1, max_end=1, n_last=-1), **sizes))


@pytest.mark.parametrize("sizes,takes", [
    ({}, 1), ({"act_dtype": 0}, 1),
    ({"vocab": 2 ** 24 - 1}, 1), ({"vocab": 2 ** 24}, 0), ({"vocab": 2 ** 31 - 1}, 0),                      # the head's bytes in 32 bits
    ({"act_dtype": 0, "vocab": 2 ** 14}, 0),                                                               # another order of sums there
    ({"head_dim": 32, "max_end": 64}, 1), ({"head_dim": 32, "max_end": 65}, 0), ({"max_end": 500}, 1),      # one page for the matrix cores' heads
    ({"inter": 256}, 0), ({"inter": 256, "n_rows": 17, "n_want": 17, "n_seqs": 17}, 1), ({"inter": 224}, 1),       # K dealt out to waves
    ({"n_heads": 17, "n_kv_heads": 1, "head_dim": 32, "n_rows": 17, "n_want": 17, "n_seqs": 17}, 0),        # more heads than a tile's columns
    ({"n_rows": 65}, 0), ({"n_want": 2}, 0), ({"hidden": 72}, 0), ({"n_layers": 17}, 0)])
def test_which_steps_the_kernel_for_small_models_takes(sizes, takes):
    lib = ctypes.CDLL(kernels.library_path())
    assert lib.tqk_small_step_takes(ctypes.byref(small_step(**sizes))) == takes


@pytest.mark.parametrize("sizes,rings", [
    ({"act_dtype": 0, "n_rows": 4, "n_want": 4, "n_seqs": 4}, 1), ({"act_dtype": 0, "n_rows": 5, "n_want": 5, "n_seqs": 5}, 0), ({"act_dtype": 0, "decode": 0}, 0),
    ({"act_dtype": 0, "vocab": 256 + 64}, 1), ({"act_dtype": 0, "vocab": 512}, 0), ({"act_dtype": 0, "vocab": 512, "n_want": 0}, 1),      # the head beside down
    ({}, 0), ({"n_heads": 3, "n_kv_heads": 1, "head_dim": 32, "hidden": 96, "inter": 224}, 1),                                        # the matrix cores' heads
    ({"n_heads": 3, "n_kv_heads": 1, "head_dim": 32, "hidden": 96, "inter": 224, "n_rows": 12, "n_want": 12, "n_seqs": 12}, 1),
    ({"n_heads": 3, "n_kv_heads": 1, "head_dim": 32, "hidden": 96, "inter": 224, "n_rows": 13, "n_want": 13, "n_seqs": 13}, 0),
    ({"head_dim": 32, "n_rows": 7, "n_want": 7, "n_seqs": 7}, 1), ({"head_dim": 32, "n_rows": 8, "n_want": 8, "n_seqs": 8}, 0),          # 14 and 16 units of attention for 14 waves
    ({"act_dtype": 0, "n_rows": 3, "n_want": 3, "n_seqs": 3, "max_end": 90}, 1), ({"act_dtype": 0, "n_rows": 4, "n_want": 4, "n_seqs": 4, "max_end": 90}, 0),
    ({"act_dtype": 0, "n_heads": 8, "n_kv_heads": 8, "head_dim": 4, "hidden": 32, "n_rows": 3, "n_want": 3, "n_seqs": 3, "max_end": 90}, 1),
    ({"act_dtype": 0, "n_heads": 8, "n_kv_heads": 8, "head_dim": 4, "hidden": 32, "n_rows": 4, "n_want": 4, "n_seqs": 4, "max_end": 90}, 0)])
def test_which_small_steps_have_their_weights_brought_into_lds(sizes, rings):
    lib = ctypes.CDLL(kernels.library_path())
    step = small_step(**sizes)
    assert lib.tqk_small_step_takes(ctypes.byref(step)) and lib.tqk_small_step_rings(ctypes.byref(step)) == rings


@pytest.mark.parametrize("sizes,rows,decode,positions,pays", [
    ({}, 33, 0, 33, 1), ({}, 40, 1, 60, 0), ({}, 24, 1, 60, 1), ({"hidden": 96, "inter": 224, "n_heads": 3, "n_kv_heads": 1, "head_dim": 32, "n_layers": 3}, 33, 0, 33, 0),
    ({"hidden": 96, "inter": 224, "n_heads": 6, "n_kv_heads": 6, "n_layers": 3, "vocab": 300}, 24, 0, 3, 0),
    ({"hidden": 96, "inter": 224, "n_heads": 6, "n_kv_heads": 1, "n_layers": 3, "vocab": 300}, 24, 0, 24, 1),
    ({"inter": 32, "n_heads": 4, "n_kv_heads": 4, "head_dim": 48, "n_layers": 4, "vocab": 97}, 20, 1, 40, 0), ({"inter": 32, "n_heads": 4, "n_kv_heads": 1, "head_dim": 48, "n_layers": 4, "vocab": 97}, 20, 1, 40, 1)])
def test_which_float32_small_steps_pay_in_one_launch(sizes, rows, decode, positions, pays):
    lib = ctypes.CDLL(kernels.library_path())
    assert lib.tqk_small_step_pays(ctypes.byref(small_step(act_dtype=0, **sizes)), rows, decode, positions) == pays


# heads, kv heads, head_dim; the sequences' new tokens; whether they are single tokens
@pytest.mark.parametrize("heads,rows,decode,pages", [
    ((4, 2, 16), [1] * 2, 1, 1), ((4, 2, 16), [1] * 16, 1, 0), ((4, 2, 16), [33], 0, 1), ((4, 4, 16), [1] * 4, 1, 0), ((5, 5, 16), [1] * 2, 1, 0), ((4, 1, 16), [1] * 40, 1, 1),
    ((8, 8, 4), [1] * 2, 1, 0), ((8, 8, 4), [1] * 16, 1, 0), ((8, 8, 4), [2] * 16, 0, 0), ((8, 8, 4), [15, 15, 15], 0, 1),
    ((2, 1, 32), [1], 1, 0), ((2, 1, 32), [8], 0, 1), ((4, 2, 32), [1], 1, 0), ((4, 2, 20), [1] * 16, 1, 0), ((8, 2, 32), [1] * 4, 1, 1),
    ((1, 1, 64), [1] * 40, 1, 0), ((1, 1, 64), [5], 0, 0), ((1, 1, 64), [16], 0, 1), ((4, 2, 64), [1], 1, 0), ((4, 2, 64), [1] * 4, 1, 1), ((3, 3, 64), [1] * 8, 1, 0)])
def test_which_float32_small_steps_have_their_attention_by_units_of_columns(heads, rows, decode, pages):
    """Steps within a page: by units where these are few beside the queries (the same bits either way, tests/test_gpu_small_step.py)."""
    lib = ctypes.CDLL(kernels.library_path())
    n_heads, n_kv, d = heads
    step = small_step(act_dtype=0, n_heads=n_heads, n_kv_heads=n_kv, head_dim=d, n_rows=sum(rows), n_want=1, n_seqs=len(rows), decode=decode, max_end=64, seq_first=10)
    for i in range(len(rows) + 1):
        step.ints[10 + i] = sum(rows[:i])
    assert lib.tqk_small_step_takes(ctypes.byref(step)) and lib.tqk_small_step_pages(ctypes.byref(step)) == pages
    step.max_end = 65
    assert lib.tqk_small_step_pages(ctypes.byref(step)) == 0


# up to 16 rows; few tiles with a group a share and with two (the last share of one, or none left over); 400 to 767 tiles either way; more
SHARES = [(16, 3584, 18944, 19), (17, 3584, 18944, 19), (100, 3584, 18944, 10), (128, 3584, 18944, 10), (160, 4096, 11008, 6), (200, 7168, 5120, 3), (300, 3584, 3584, 4), (500, 4608, 3584, 4),
          (64, 37888, 3584, 4), (128, 37888, 3584, 4), (1000, 4608, 3584, 4), (1000, 3584, 3584, 1), (1000, 3584, 18944, 1), (300, 37888, 3584, 1), (2000, 4608, 3584, 1), (40, 1024, 1024, 1)]


@pytest.mark.parametrize("m,n,k,shares", SHARES)
def test_how_many_blocks_share_a_float32_products_k(m, n, k, shares):
    lib = kernels.library()
    assert lib.tqk_gemm_f32_shares(m, n, k) == shares
    assert lib.tqk_gemm_scratch_bytes(0, 0, 0, 0, m, n, k) == (0 if shares == 1 else -(-k // 1024) * m * n * 4)


def test_the_scratch_of_float32_products_is_bounded():
    """128 MB from 512 tiles of 64 rows by 128 features on, none from 768 on; fewer tiles bound it by their own size, 16 MB for each 1024 of K."""
    lib = kernels.library()
    for k in (1024, 2052, 3584, 11008, 18944, 65536):
        for rows in range(64, 1601, 128):
            for features in (2048, 3840, 5120, 37888):
                got, tiles = lib.tqk_gemm_scratch_bytes(0, 0, 0, 0, rows, features, k), -(-rows // 64) * -(-features // 128)
                if tiles * -(-k // 1024) >= 256 and rows > 32:         # (the largest tiles are taken)
                    assert got <= (0 if tiles >= 768 else 128 << 20 if tiles >= 512 else tiles * 64 * 128 * 4 * -(-k // 1024)), (rows, features, k)
