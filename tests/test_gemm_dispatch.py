"""The GEMM dispatch (trlm_gemm.c) without a GPU: the file is compiled against
stand-ins of hip_backend.h's calls that write down what would be launched.

  - trlm_gemm_last_variant names the kernel and split count that were
    launched, and trlm_gemm_plan_ex foretells them, over shapes, layouts and
    both kinds of engine;
  - at most one 64x64 workgroup per CU (256) takes the fp32 tile, beyond it
    the split products;
  - the gate/up product with its SwiGLU has the same lines: the small kernel,
    the fp32 tile up to 256 workgroups, then the split products;
  - with 32 MiB for the partials, as trlm_gemm_noalloc has, exactly the products
    that its documentation names run with fewer splits than planned;
  - an engine kept to fp32 launches no split product, and neither does any
    engine for row statistics or column sums, which those kernels do not form."""
import os
import random
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM_INC = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include")
pytestmark = pytest.mark.skipif(not os.path.exists(os.path.join(ROCM_INC, "hip", "hip_runtime_api.h")),
                                reason="HIP headers not present")

HARNESS = r"""
#include "trlm_gemm.c"
static int xlookups;
hipFunction_t hip_get_kernel(HipCtx* c, const char* name) {
    (void)c;
    xlookups += !strncmp(name, "k_xgemm", 7);
    return (hipFunction_t)strdup(name);
}
void hip_launch(hipFunction_t f, u32 gx, u32 gy, u32 gz, u32 bx, u32 by, u32 bz, u32 shared, void** args) {
    (void)gy; (void)bx; (void)by; (void)bz; (void)shared; (void)args;
    printf("%s %u %u ", (const char*)f, gx, gz);
}
hipDeviceptr_t hip_alloc(u64 bytes) { (void)bytes; return (hipDeviceptr_t)0x70000000; }
void hip_free(hipDeviceptr_t p) { (void)p; }
hipStream_t hip_current_stream(void) { return NULL; }
void trlm_noalloc_setup(i32 device) { (void)device; }
int main(void) {
    HipCtx ctx;
    memset(&ctx, 0, sizeof(ctx));
    TrlmGemm* e[2] = { trlm_gemm_create_fp32(&ctx), trlm_gemm_create_fp32(&ctx) };
    if (xlookups) return 1;                        /* a trainer's engines look up what they can launch */
    e[0] = trlm_gemm_create(&ctx);
    int fp32, ta, tb, M, N, K, glu_F, aligned, splits, sums;
    unsigned long long ws;
    while (scanf("%d %d %d %d %d %d %d %d %llu %d", &fp32, &ta, &tb, &M, &N, &K, &glu_F, &aligned, &ws, &sums) == 10) {
        TrlmGemmExtra x;
        memset(&x, 0, sizeof(x));
        if (sums && tb) { x.stats = (hipDeviceptr_t)0x800000; x.stats_cap = 1 << 20; }
        if (sums && !tb) x.csum = (hipDeviceptr_t)0x900000;
        x.glu_h = glu_F ? (hipDeviceptr_t)0x600000 : NULL;
        x.glu_F = glu_F;
        const int la = ((ta ? M : K) + 3) / 4 * 4 + !aligned, lb = ((tb ? K : N) + 3) / 4 * 4 + !aligned;
        trlm_gemm_ws(e[fp32], ta, tb, (hipDeviceptr_t)0x100000, (hipDeviceptr_t)0x200000, (hipDeviceptr_t)0x300000,
                     M, N, K, la, lb, N, 1, 0, 0, 0, 1.0f, 0.0f, NULL, NULL, N, glu_F || sums ? &x : NULL,
                     ws ? (hipDeviceptr_t)0x400000 : NULL, ws);
        const char* name = trlm_gemm_last_variant(e[fp32], &splits);
        printf("| %s %d ", name, splits);
        name = trlm_gemm_plan_ex(ta, tb, M, N, K, 1, fp32, glu_F, &splits);
        printf("| %s %d\n", name, splits);
    }
    return 0;
}
"""


@pytest.fixture(scope="module")
def dispatch(tmp_path_factory):
    """calls [(fp32, ta, tb, M, N, K, glu_F, aligned, fixed workspace floats
    [, row statistics (NT) or column sums])] ->
    [(launches [(kernel, grid x, grid z)], (reported, splits), (planned, splits))]"""
    d = tmp_path_factory.mktemp("dispatch")
    (d / "h.c").write_text(HARNESS)
    csrc = os.path.join(ROOT, "turkce-llm_amd", "csrc")
    subprocess.run(["gcc", "-std=c11", "-O1", "-D__HIP_PLATFORM_AMD__", "-D_DEFAULT_SOURCE", "-I" + csrc,
                    "-I" + os.path.join(ROOT, "include"), "-I" + ROCM_INC, str(d / "h.c"), "-o", str(d / "h"),
                    "-L" + os.path.join(ROCM_INC, "..", "lib"), "-Wl,-rpath," + os.path.join(ROCM_INC, "..", "lib"),
                    "-lamdhip64"], check=True)

    def run(calls):
        text = "\n".join(" ".join(str(int(v)) for v in (*c, 0)[:10]) for c in calls) + "\n"
        out = subprocess.run([str(d / "h")], input=text, check=True, capture_output=True, text=True).stdout
        res = []
        for line in out.splitlines():
            a, b, c = [part.split() for part in line.split("|")]
            res.append(([(a[i], int(a[i + 1]), int(a[i + 2])) for i in range(0, len(a), 3)], (b[0], int(b[1])),
                        (c[0], int(c[1]))))
        assert len(res) == len(calls)
        return res

    return run


def drawn(n, seed):
    rng = random.Random(seed)
    size = lambda hi: int(round(2 ** rng.uniform(0, hi)))
    return [(rng.randint(0, 1), *rng.choice([(0, 0), (0, 1), (1, 0)]), size(13), size(14), size(13), 0,
             rng.random() < 0.75, 0) for _ in range(n)]


def test_reported_and_planned_names_are_the_launched_kernels(dispatch):
    calls = drawn(4000, 1) + [(fp32, 0, 0, M, 2 * F, K, F, 1, 0) for fp32 in (0, 1) for M in (1, 100, 512, 700, 8192)
                              for F, K in ((32, 32), (1024, 384), (2048, 768))]
    families = set()
    for call, (launches, (name, splits), plan) in zip(calls, dispatch(calls)):
        kernel, _, gz = launches[0]
        assert name == kernel, call
        assert gz == splits and len(launches) == (2 if splits > 1 else 1), call
        assert not (call[0] and kernel.startswith("k_xgemm")), call
        if call[7]:
            assert plan == (name, splits), call
        families.add((call[0], kernel.rsplit("_", 1)[0] if call[6] else kernel.split("_")[1]))
    assert {(0, "gemm"), (0, "xgemm"), (0, "smallgemm"), (1, "gemm"), (1, "smallgemm")} <= families


def test_lone_64x64_workgroups_take_the_fp32_tile(dispatch):
    seen = {True: 0, False: 0}
    for call, (launches, _, _) in zip(drawn(4000, 2), dispatch(drawn(4000, 2))):
        kernel, gx, gz = launches[0]
        if not call[0] and call[7] and kernel.endswith("_64x64_k32"):
            lone = gx * gz <= 256
            assert kernel.startswith("k_gemm_" if lone else "k_xgemm_"), (call, launches)
            seen[lone] += 1
    assert min(seen.values()) >= 50, seen


@pytest.mark.parametrize("M,F,K,want", [
    (1, 32, 32, "k_smallgemm_nn_glu"), (100, 1024, 384, "k_smallgemm_nn_glu"), (256, 1024, 384, "k_smallgemm_nn_glu"),
    (257, 1024, 384, "k_gemm_nn_64x64_k32_glu"), (512, 1024, 384, "k_gemm_nn_64x64_k32_glu"),
    (513, 1024, 384, "k_xgemm_nn_64x64_k32_glu"), (8192, 1024, 384, "k_xgemm_nn_128x128_glu"),
    (8192, 1056, 384, "k_xgemm_nn_64x64_k32_glu"), (64, 2048, 768, "k_smallgemm_nn_glu"),
    (65, 2048, 768, "k_gemm_nn_64x64_k32_glu"), (64, 1024, 2048, "k_gemm_nn_64x64_k32_glu")])
def test_swiglu_kernels(dispatch, M, F, K, want):
    free, kept = dispatch([(fp32, 0, 0, M, 2 * F, K, F, 1, 0) for fp32 in (0, 1)])
    tile = {"s": 32}.get(want[2], 128 if "128" in want else 64)
    assert free[0] == [(want, -(-M // tile) * -(-2 * F // tile), 1)]
    assert kept[0][0][0] == (want if "smallgemm" in want else "k_gemm_nn_64x64_k32_glu")


def test_products_whose_partials_exceed_32_mib(dispatch):
    N, D, F, V, room = 8192, 384, 1024, 31769, (32 << 20) // 4
    shapes = {"QKV fwd": (0, 0, N, 3 * D, D), "out fwd": (0, 0, N, D, D), "gate/up fwd": (0, 0, N, 2 * F, D),
              "down fwd": (0, 0, N, D, F), "head fwd": (0, 1, N, V, D), "QKV dX": (0, 1, N, D, 3 * D),
              "out dX": (0, 1, N, D, D), "gate/up dX": (0, 1, N, D, 2 * F), "down dX": (0, 1, N, F, D),
              "head dX": (0, 0, N, D, V), "QKV dW": (1, 0, D, 3 * D, N), "out dW": (1, 0, D, D, N),
              "gate/up dW": (1, 0, D, 2 * F, N), "down dW": (1, 0, F, D, N), "head dW": (1, 0, V, D, N)}
    fewer = set()
    for (name, s), (_, (_, ran), (_, planned)) in zip(shapes.items(),
                                                      dispatch([(0, *s, 0, 1, room) for s in shapes.values()])):
        M, Nc = s[2], s[3]
        assert ran == 1 or ran * M * Nc <= room, name
        if ran < planned:
            assert planned * M * Nc > room, name
            fewer.add(name)
    assert fewer == {"gate/up dX", "gate/up dW", "down dW", "head dX", "head dW"}


def test_sums_are_formed_by_the_fp32_kernels(dispatch):
    calls = [(fp32, ta, tb, M, 2048, 8192, 0, aligned, 0, 1) for fp32 in (0, 1) for ta, tb in ((0, 1), (1, 0), (0, 0))
             for M in (64, 384, 8192) for aligned in (0, 1)]
    for call, (launches, (name, _), _) in zip(calls, dispatch(calls)):
        assert name.startswith("k_gemm_") and launches[0][0] == name, call
