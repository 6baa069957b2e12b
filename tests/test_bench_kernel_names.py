"""Every kernel name bench.py hands to q38_kernel_timer_start is one the
library's lookup accepts, and every projection kernel the library may launch
is one bench.py times (CPU only: the library's names are read from its
source), so that no measurement fails, or leaves a part out, at run time."""
import os
import re

import bench

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HOST = os.path.join(ROOT, "qwen3.8_27b_in_rust_amd", "csrc", "host", "q38_attn.cpp")


def _timer_names():
    src = open(HOST).read()
    body = src[src.index("int q38_kernel_timer_start("):]
    body = body[:body.index("\n}\n")]
    names = set(re.findall(r'name == "(q38_[a-z0-9_]+)"', body))
    table = src[src.index("constexpr GemvType kGemv[] = {"):]
    table = table[:table.index("};")]
    names |= set(re.findall(r'"(q38_[a-z0-9_]+)"', table))
    return names


def _accepts(names, name):
    return name in names


def test_bench_timer_names_are_known():
    names = _timer_names()
    used = {bench.DECODE_KERNEL, "q38_attn_decode_merge", "q38_gdn_step_rows", "q38_noop", "q38_gdn_decode",
            "q38_attn_prefill_mfma", "q38_prefill_merge", "q38_kv_split_mfma", "q38_attn_decode_split_many",
            "q38_gdn_pre", "q38_gdn_post", "q38_copy_f32"}
    for ty in bench.GEMV_KERNELS:
        used.update(bench._q8k_kernels(ty))
    for ty in bench.F32_PATH_TYPES:
        used.update(bench._f32_path_kernels(ty))
    unknown = sorted(n for n in used if not _accepts(names, n))
    assert not unknown, unknown


def test_bench_literal_kernel_names_are_known():
    """Every literal "q38_..." kernel name passed to kernel_timer_start in
    bench.py."""
    names = _timer_names()
    src = open(os.path.join(ROOT, "bench.py")).read()
    lits = set(re.findall(r'kernel_timer_start\("(q38_[a-z0-9_]+)"', src))
    for tup in re.findall(r'for name in \(([^)]*)\)', src):
        lits |= set(re.findall(r'"(q38_[a-z0-9_]+)"', tup))
    assert lits, "no literal names found"
    assert not sorted(n for n in lits if not _accepts(names, n))


def test_library_projection_kernels_are_timed():
    """Every form in the library's table of Q8_K kernels, of its weight type,
    and every f32-path kernel."""
    src = open(HOST).read()
    table = src[src.index("constexpr GemvType kGemv[] = {"):]
    rows = [re.findall(r'"(q38_[a-z0-9_]+)"', r) for r in table[:table.index("};")].split("\n") if '"q38_' in r]
    by_gemv = {bench.GEMV_KERNELS[ty]: set(bench._q8k_kernels(ty)) for ty in bench.GEMV_KERNELS}
    assert len(rows) == len(by_gemv)
    for names in rows:
        assert set(names) == by_gemv[names[0]], names[0]
    f32 = {n for n in _timer_names() if n.startswith(("q38_gemv_f32_", "q38_gemm_f32"))}
    assert f32 == {n for ty in bench.F32_PATH_TYPES for n in bench._f32_path_kernels(ty)}


class _TwoForms:
    """A context whose projection call launches the 128 x 256 tiles (3 ms) and,
    for each of two matrices, a split-block form (1 ms)."""
    LAUNCHES = {"q38_gemm_wide_q8k_q4k": (3.0, 1), "q38_gemm_ks4_q8k_q4k": (1.0, 2)}

    def __init__(self):
        self.name, self.calls = None, 0

    def kernel_timer_start(self, name, max_launches):
        self.name, self.calls = name, 0

    def gemv_q8_k(self, *args):
        self.calls += 1

    def kernel_timer_stop(self):
        ms, n = self.LAUNCHES.get(self.name, (0.0, 0))
        return ms * n * self.calls, n * self.calls


def test_a_call_of_two_forms_is_timed_whole():
    kern, ms = bench._timed_projection(_TwoForms(), 12, 17408, 5120, None, None, 3001, None, reps=4)
    assert set(kern.split(" + ")) == set(_TwoForms.LAUNCHES)
    assert ms == 5.0
