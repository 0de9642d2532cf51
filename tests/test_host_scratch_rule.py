"""The pinned host scratch's rules (eakv_amd/csrc/cache.c) on the CPU: the file is
compiled with a counting device layer in place of the HIP one."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "eakv_amd", "csrc")

PROGRAM = r"""
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include "internal.h"

static int mallocs, h2d, kernels;
int eakvd_host_malloc(void **p, size_t n) { mallocs++; *p = malloc(n); return 0; }
int eakvd_host_free(void *p) { free(p); return 0; }
int eakvd_memcpy_h2d_async(void *d, const void *s, size_t n, void *st)
{ (void)st; h2d++; memcpy(d, s, n); return 0; }
int eakvd_copy_in(void *d, const void *s, size_t n, void *st)
{ (void)st; kernels++; memcpy(d, s, n); return 0; }

int main(int argc, char **argv)
{
    eakv_cache_t c;
    memset(&c, 0, sizeof(c));
    if (argc == 2) {                     /* a buffer that grows by 128 bytes a call */
        size_t need = 65536;
        for (int i = 0; i < 4096; i++, need += 128) {
            void *p = NULL;
            if (eakvi_pinned(&c, need, &p) || !p || c.pin_bytes < need) return 2;
            memset(p, 1, need);
        }
        printf("%d %zu %zu\n", mallocs, c.pin_bytes, need - 128);
        return 0;
    }
    /* one input of argv[1] bytes, read once or (argv[2] = 0) by many blocks */
    size_t n = (size_t)atoll(argv[1]);
    char *src = malloc(n), *dev = calloc(1, n);
    for (size_t i = 0; i < n; i++) src[i] = (char)(i * 31 + 7);
    eakvi_bounce bo;
    const void *k = NULL;
    eakvi_bounce_begin(&c, n, 64, &bo);
    if (eakvi_bounce_in(&bo, dev, src, n, atoi(argv[2]), NULL, &k)) return 2;
    if (memcmp(k, src, n)) return 3;
    printf("%s %d %d\n", k == dev ? "device" : k == bo.pin ? "scratch" : "?", h2d, kernels);
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    cc = shutil.which("gcc")
    if not cc:
        pytest.skip("gcc not available")
    d = tmp_path_factory.mktemp("scratch")
    (d / "main.c").write_text(PROGRAM)
    exe = str(d / "main")
    subprocess.run([cc, "-std=c11", "-O1", "-I", SRC, "-I", os.path.join(ROOT, "include"),
                    str(d / "main.c"), os.path.join(SRC, "cache.c"), "-o", exe,
                    "-Wl,--unresolved-symbols=ignore-all"], check=True)
    return exe


def run(program, *args):
    return subprocess.run([program, *map(str, args)], check=True, capture_output=True,
                          text=True).stdout.split()


MIB = 1 << 20


@pytest.mark.parametrize("n,once,where", [
    (4, 1, ("scratch", 0, 0)), (4, 0, ("device", 0, 1)),
    (MIB, 1, ("scratch", 0, 0)), (MIB, 0, ("device", 0, 1)),
    (MIB + 4, 1, ("device", 1, 0)), (MIB + 4, 0, ("device", 1, 0)),
    (4 * MIB - 256, 1, ("device", 1, 0)), (4 * MIB + 4, 1, ("device", 1, 0))])
def test_where_an_input_is_read(program, n, once, where):
    """In place up to 1 MiB; by a copy above, from the scratch up to 4 MiB with
    the result and from the caller's memory beyond."""
    place, h2d, kernels = run(program, n, once)
    assert (place, int(h2d), int(kernels)) == where


def test_growing_needs_allocate_rarely(program):
    """A decode loop's scores and weights grow with every token: 4096 calls that
    each need 128 bytes more, 64 KiB to 576 KiB, allocate at most once per
    quarter (1.25^10 > 9), and hold at most a quarter more than needed."""
    mallocs, held, need = map(int, run(program, "grow"))
    assert 1 <= mallocs <= 11
    assert need <= held <= need + need // 4
