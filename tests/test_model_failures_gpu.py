"""The decode engine when a HIP call fails: a small shared object, loaded
ahead of the HIP runtime in a process of its own, counts device allocations
and lets a chosen allocation or one device-to-host copy return an error
without being made.  Every kernel runs and ends as usual."""
import os
import subprocess
import sys
import textwrap

import pytest

pytestmark = pytest.mark.gpu

SHIM = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <link.h>
#include <stdlib.h>
#include <string.h>
int shim_mallocs, shim_fail_malloc, shim_fail_d2h, shim_copies;
static int find(struct dl_phdr_info *i, size_t n, void *p) {
    (void)n;
    if (!strstr(i->dlpi_name, "libamdhip64")) return 0;
    *(void **)p = dlopen(i->dlpi_name, RTLD_LAZY | RTLD_NOLOAD);
    return 1;
}
static void *real(const char *name) {
    void *h = 0;
    dl_iterate_phdr(find, &h);
    void *f = h ? dlsym(h, name) : 0;
    if (!f) abort();
    return f;
}
int hipMalloc(void **p, size_t n) {
    static int (*f)(void **, size_t);
    if (!f) f = (int (*)(void **, size_t))real("hipMalloc");
    if (++shim_mallocs == shim_fail_malloc) { *p = 0; return 2; }     /* hipErrorOutOfMemory */
    return f(p, n);
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *st) {
    static int (*f)(void *, const void *, size_t, int, void *);
    if (!f) f = (int (*)(void *, const void *, size_t, int, void *))real("hipMemcpyAsync");
    shim_copies++;
    if (kind == 2 && shim_fail_d2h) { shim_fail_d2h = 0; return 999; } /* hipErrorUnknown */
    return f(d, s, n, kind, st);
}
"""

PRELUDE = """
import ctypes as C, sys
shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
v = lambda n: C.c_int.in_dll(shim, n)
import numpy as np
import libinferbit_amd as L
from libinferbit_amd import ibf
from libinferbit_amd._lib import IbhError
from libinferbit_amd.model import Model
cfg = dict(ibf.TINYLLAMA, num_layers=2, hidden_size=256, num_heads=4, num_kv_heads=2, head_dim=64,
           intermediate_size=512, vocab_size=1000, max_context_length=200)
ibf.write_synthetic(sys.argv[2], cfg, seed=31)
toks = np.random.default_rng(7).integers(0, 1000, 64).astype(np.int32)
same = lambda a, b: np.array_equal(np.asarray(a).view(np.uint32), np.asarray(b).view(np.uint32))
err = lambda: L.lib().ibh_last_error()
"""


def run(tmp_path, code):
    src, so = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", str(so), str(src), "-ldl"], check=True)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-u", "-c", PRELUDE + textwrap.dedent(code), str(so), str(tmp_path / "m.ibf")],
                       cwd=root, capture_output=True, text=True, timeout=100)
    print(r.stdout[-2000:], r.stderr[-4000:], flush=True)
    assert r.returncode == 0 and "checked" in r.stdout


def test_load_without_memory_for_batches(tmp_path):
    """A model whose batch buffers find no memory loads without a word, steps
    through its prompts without asking for them again, and batches once a
    forward_positions call has found them."""
    run(tmp_path, """
        Model(sys.argv[2]).close()                           # and the library's own buffers
        n = v("shim_mallocs").value
        ok = Model(sys.argv[2])
        per = v("shim_mallocs").value - n
        assert per > 10
        n += 2 * per
        v("shim_fail_malloc").value = n                      # the last allocation of the next load
        assert err() in (None, b"")
        m = Model(sys.argv[2])
        assert v("shim_mallocs").value == n
        assert err() in (None, b""), err()
        for _ in range(3):
            assert same(m.forward(toks[:9]), ok.forward(toks[:9]))
        assert v("shim_mallocs").value == n
        assert same(m.forward_positions(toks[:5]), ok.forward_positions(toks[:5]))
        assert v("shim_mallocs").value == n + 1
        assert same(m.forward(toks[:9]), ok.forward(toks[:9]))
        # fast mode takes its attention partials when it is chosen, or does without
        n = v("shim_mallocs").value
        ok.set_exact(False)
        v("shim_fail_malloc").value = n + 2
        m.set_exact(False)
        assert v("shim_mallocs").value == n + 2 and err() in (None, b"")
        assert same(m.forward_positions(toks[:12]), ok.forward_positions(toks[:12]))
        assert same(m.forward(toks[:9]), ok.forward(toks[:9]))
        assert v("shim_mallocs").value == n + 2
        print("checked")
        """)


def test_position_after_a_failed_call(tmp_path):
    """A call whose pass ran but whose logits did not arrive leaves the length
    as it was, and what follows starts from that length: the same results as
    from a model that never saw it, also at the end of the context."""
    run(tmp_path, """
        def fails(f):
            v("shim_fail_d2h").value = 1
            try:
                f()
            except IbhError:
                assert v("shim_fail_d2h").value == 0         # the copy was reached and failed
                return
            raise SystemExit("the copy did not fail")

        a, b = Model(sys.argv[2]), Model(sys.argv[2])
        for m in (a, b):
            m.forward(toks[:20])
        for n in (5, 32, 1):
            fails(lambda: a.forward_positions(toks[:n]))
            assert a.kv_length() == b.kv_length()
            assert same(a.forward_positions(toks[3:7]), b.forward_positions(toks[3:7]))
            assert same(a.forward(toks[9:10]), b.forward(toks[9:10]))
        # up to the last position of the context
        while b.kv_length() < 199:
            n = min(32, 199 - b.kv_length())
            fails(lambda: a.forward_positions(toks[:n]))
            assert same(a.forward_positions(toks[:n]), b.forward_positions(toks[:n]))
        fails(lambda: a.forward_positions(toks[:1]))
        assert same(a.forward_positions(toks[:1]), b.forward_positions(toks[:1]))
        assert a.kv_length() == b.kv_length() == 200
        print("checked")
        """)
