"""What the class layer asks of the C ABI and in which order, on the CPU: small programs over libzkllm_prover.so that define the
entry points they reach themselves (a program's own definitions come before the kernel library's).  No GPU needed."""
import os
import subprocess

import pytest

from zkhelp import ROOT

PKG = os.path.join(ROOT, "zkllm-ccs2024_amd")

# device memory is host memory here; `events` holds the calls that a test looks at
ABI = r"""
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <thread>
#include <vector>
#include "zksoftmax.hpp"
static std::vector<std::string> events;
static std::vector<const void*> job;          // what an opened job was given to read
static std::atomic<int> frees{0}, reads{0};
static int ready = -1;                       // whether the last opened job's queries were
extern "C" {
const char* zk_last_error() { return "refused"; }
int zk_malloc(void** p, size_t n) { *p = calloc(1, n + 64); return 0; }
int zk_free(void* p) {
    ++frees;
    for (const void* q : job) if (p == q) events.push_back("free of the job's");
    free(p);
    return 0;
}
int zk_sync(void*) { events.push_back("wait"); return 0; }
int zk_upload(void* d, const void* s, size_t n, void*) { memcpy(d, s, n); return 0; }
int zk_memcpy_d2h(void* d, const void* s, size_t n, void*) {
    ++reads;
    events.push_back("wait");
    std::this_thread::sleep_for(std::chrono::milliseconds(50));
    memcpy(d, s, n);
    return 0;
}
int zk_range_table(void*, int32_t, uint32_t, uint32_t, void*) { return 0; }
int zk_fr_from_i32(void*, const void*, size_t, void*) { return 0; }
int zk_softmax_table(void*, double, double, uint32_t, void*) { return 0; }
int zk_fr_pad_from(void*, const void*, size_t, size_t, const void*, void*) { return 0; }
int zk_fr_fold_prepare(void** p, const void*, size_t, void*) { events.push_back("wait"); *p = malloc(4); return 0; }
int zk_fr_fold_prepare_queue(void** p, void* flag, const void*, size_t, void*) { *p = malloc(4); memset(flag, 0, 4); return 0; }
int zk_fr_fold_prepared_new(void** p, void** ints, size_t, void*) { *p = malloc(4); *ints = *p; return 0; }
const void* zk_fr_fold_prepared_ints(const void* p) { return p; }
int zk_fr_fold_prepared_free(void* p) { return zk_free(p); }
int zk_fr_add_mul_s(void*, const void*, const void*, const uint32_t*, size_t, void*) { return 0; }
int zk_fr_copy_add_first(void*, const void*, const uint32_t*, size_t, void*) { return 0; }
int zk_fr_gather(void*, const void*, const void*, size_t, void*) { return 0; }
int zk_fr_gather_ints(void*, void*, const void*, const void*, const void*, size_t, void*) { return 0; }
int zk_i32_pad_from(void*, const void*, size_t, size_t, const void*, int32_t, void*) { return 0; }
int zk_lookup_ints_suffice(size_t, size_t) { return 0; }
int zk_lookup_multiplicities(void*, void*, const void*, const void*, const void*, int32_t, uint32_t, size_t, uint32_t, int, void*) { events.push_back("counted"); return 0; }
int zk_lookup_multiplicities_begin(void** c, void*, void*, const void*, const void*, const void*, int32_t, uint32_t, size_t, uint32_t, void*) { events.push_back("count begun"); *c = malloc(4); return 0; }
int zk_lookup_multiplicities_end(void* c) { free(c); return 0; }
int zk_lookup_open(void** o, const void*, const uint32_t*, size_t, void*) { *o = malloc(4); return 0; }
int zk_lookup_open_drop(void* o) { events.push_back("drop"); free(o); return 0; }
int zk_lookup_prove_begin_opened(void**, void*, const void* S, const void* Si, const void* So, const void* Soi, const void* mi, const uint32_t*, const void* T, const void* m, int32_t,
                                 const uint32_t*, const uint32_t*, const uint32_t*, size_t, size_t, int, int queries_ready, int, void*) {
    ready = queries_ready;
    for (const void* p : {S, Si, So, Soi, mi, T, m}) if (p) job.push_back(p);
    events.push_back("begin");
    return 1;
}
}
"""


def run(tmp_path, name, body):
    src = tmp_path / (name + ".cpp")
    src.write_text(ABI + body)
    exe = str(tmp_path / name)
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-rdynamic", "-I" + os.path.join(PKG, "host"), str(src), "-o", exe, "-L" + PKG, "-lzkllm_prover", "-lzkllm_hip",
                    "-Wl,-rpath," + PKG], check=True)
    return subprocess.run([exe], check=True, capture_output=True, text=True, timeout=60).stdout.splitlines()


def test_first_questions_for_an_int32_form_from_two_threads_settle_it_once(tmp_path):
    """A tensor whose producer has not been asked yet whether every element fits: the flag is read and given back once, and both threads get the form."""
    out = run(tmp_path, "settle", r"""
int main() {
    FrTensor t(8);
    t.keep_for_folds_queued();
    const int before = frees;
    const void* got[2];
    std::thread a([&] { got[0] = t.kept_ints(); }), b([&] { got[1] = t.kept_ints(); });
    a.join(); b.join();
    printf("%d\n%d\n%d\n", (int)reads, frees - before, got[0] && got[0] == got[1]);
    fflush(stdout);
    _Exit(0);
}
""")
    assert out == ["1", "1", "1"]


def test_failed_proof_on_an_opened_table_lets_its_tensors_go_behind_the_job(tmp_path):
    """zk_lookup_prove_begin_opened may have queued kernels before it fails: what they read is freed only when the opened job has been dropped, which waits for them."""
    out = run(tmp_path, "order", r"""
int main() {
    FrTensor values(4), queries(6);
    tLookupRangeMapping table(-2, 4, values);
    const vector<Fr_t> u(3), v(3);
    events.clear();
    try { table.map_and_prove_begin(queries, Fr_t{}, Fr_t{}, Fr_t{}, u, v); } catch (const std::exception&) { events.push_back("thrown"); }
    for (auto& e : events) puts(e.c_str());
    fflush(stdout);
    _Exit(0);
}
""")
    assert out[-1] == "thrown" and out[out.index("begin") + 1] == "drop"
    assert out.count("free of the job's") >= 3          # padded queries and outputs, the combined table


def test_constructor_of_a_mapping_table_leaves_nothing_queued_or_unsettled(tmp_path):
    """A table that a caller has constructed is complete and only read from then on, whatever stream or thread goes on with it; one made with `queued` waits for nothing."""
    out = run(tmp_path, "made", r"""
int main() {
    FrTensor values(4);
    tLookupRangeMapping table(-2, 4, values);
    printf("%d\n%d\n", (int)events.size(), table.mapped_vals.fold_cache->unchecked == nullptr);
    events.clear();
    tLookupRangeMapping queued(-2, 4, values, tLookupRangeMapping::queued);
    printf("%d\n", (int)events.size());
    fflush(stdout);
    _Exit(0);
}
""")
    assert out == ["1", "1", "0"]


def test_mapping_that_waits_for_its_check_at_once_counts_in_one_call(tmp_path):
    """An event for a check that is asked for in the next line costs more than the check."""
    out = run(tmp_path, "counts", r"""
int main() {
    FrTensor values(4), queries(6);
    tLookupRangeMapping table(-2, 4, values);
    events.clear();
    (void)table(queries);
    for (auto& e : events) if (e[0] == 'c') puts(e.c_str());
    fflush(stdout);
    _Exit(0);
}
""")
    assert out == ["counted"]


def test_constructor_of_a_softmax_leaves_its_tables_settled(tmp_path):
    out = run(tmp_path, "softmax", r"""
struct Softmax : zkSoftmax { using zkSoftmax::zkSoftmax; using zkSoftmax::other_segments; };
int main() {
    Softmax s({4, 4, 4}, 1, 1, 1, {1.0}, 4, 4, 4, 1);
    for (auto& t : s.other_segments) printf("%d\n", t.mapped_vals.fold_cache->unchecked == nullptr);
    fflush(stdout);
    _Exit(0);
}
""")
    assert out == ["1", "1"]


@pytest.mark.parametrize("log_queries,log_table,more,ahead", [(23, 16, 1, 1), (24, 15, 1, 1), (24, 16, 1, 0), (24, 20, 1, 0), (25, 16, 1, 0), (24, 16, 0, 1), (10, 4, 1, 1)])
def test_rounds_of_a_large_job_wait_for_the_counting_where_more_is_queued_behind_it(tmp_path, log_queries, log_table, more, ahead):
    out = run(tmp_path, "ahead", r"""
int main() {
    FrTensor S(1u << %d);
    tLookupRange table(0, 1u << %d);
    const vector<Fr_t> u(%d), v(%d);
    std::unique_ptr<FrTensor> m;
    try { table.count_and_prove_begin(S, m, true, Fr_t{}, Fr_t{}, u, v, true, %d); } catch (const std::exception&) {}
    printf("%%d\n", ready);
    fflush(stdout);
    _Exit(0);
}
""" % (log_queries, log_table, log_queries, log_queries, more))
    assert out == [str(ahead)]
