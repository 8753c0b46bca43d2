"""How fp32 products are cut for the bf16 matrix cores, on the CPU through the built library
(tests/split_plan/split_plan.cpp): what the kernels assume of alignments, beta, slices and workspace
holds for every part of every cut."""
import os
import re
import subprocess

import pytest

from test_gemm_split_gpu import CUTS

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DIR = os.path.join(ROOT, "tests", "split_plan")


@pytest.fixture(scope="module")
def plan():
    subprocess.run(["make", "-s", "-C", DIR], check=True, capture_output=True)
    return os.path.join(DIR, "_build", "split_plan")


def test_every_part_of_every_cut_keeps_the_kernels_assumptions(plan):
    r = subprocess.run([plan], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-4000:]
    assert r.stdout.strip().endswith("0 violations")
    seen = {k: int(v) for k, v in re.findall(r"(\w+) (\d+)", r.stdout.splitlines()[0])}
    assert all(v > 500 for v in seen.values()), seen  # every form of cut was walked


@pytest.mark.parametrize("M,N,K,batch,layout,taken", [(130, 2567, 2071, 17, "tt", False), (130, 2568, 2072, 17, "tt", True),
                                                      (777, 1234, 4099, 1, "tn", True), (192, 1673, 3070, 14, "tt", False)])
def test_packing_off_16_bytes_is_priced(plan, M, N, K, batch, layout, taken):
    """Large operands with K-contiguous rows off 16 bytes are packed at a lower rate: 17 x 130 x 2567 x 2071 TT
    took 594 us on the bf16 cores, 466 on the fp32 ones; 14 x 192 x 1673 x 3070 TT 465 and 408."""
    out = subprocess.run([plan, *map(str, (M, N, K, batch, layout, 0))], capture_output=True, text=True).stdout
    assert (out.strip() != "none") == taken


def test_each_gate_word_is_written_by_one_kernel_and_tested_by_later_ones():
    src = open(os.path.join(ROOT, "go-nngpu_amd", "csrc", "gemm_split.hip")).read()
    pack, product = src.split("split_pack_kernel(", 1)[1].split("gemm_split_kernel(", 1)
    product = product.split("hipError_t launch_tile", 1)[0]
    assert re.findall(r"gate->(\w+)", pack) == ["packed"]
    # the product kernel writes the one word and tests the gate through the function above only
    assert re.findall(r"gate->(\w+)", product) == ["multiplied"]
    assert re.findall(r"\w+\(\*p\.gate|\*p\.gate", product) == ["split_product_skipped(*p.gate"]


@pytest.mark.parametrize("M,N,K,batch,layout,gap,form", CUTS)
def test_gpu_cases_reach_the_cuts_they_name(plan, M, N, K, batch, layout, gap, form):
    out = subprocess.run([plan, *map(str, (M, N, K, batch, layout, gap))], capture_output=True, text=True).stdout
    m = re.match(r"nb (\d+) kc (\d+) raw (\d) S (\d+)", out)
    assert m, out
    nb, kc, raw, S = map(int, m.groups())
    assert {"batch": 1 < nb < batch, "single": nb == 1 < batch, "k": kc < K}[form.split("-")[0]]
    assert raw == form.endswith("raw")


# Products whose time a kernel of their own brings down: dtype, layout, M, N, K, kernel (on MI355X the next best took
# the factor in the comment)
ROUTES = [("f32", "nn", 1, 32768, 255, "gemv"),  # 3.5
          ("f32", "nn", 4, 65536, 128, "gemv"),  # 1.8
          ("f16", "nn", 2, 32768, 128, "gemv"),  # 2.0
          ("f32", "nn", 1, 16384, 512, "gemv"),  # 1.17
          ("f16", "nn", 1, 65536, 256, "gemv"),  # 1.4
          ("f16", "nt", 1, 65536, 256, "rows-4"),  # 3.2 (16 waves)
          ("f16", "nt", 8, 32768, 512, "rows-4"),  # 1.7 (16 waves)
          ("f32", "nt", 2, 32768, 256, "rows-4"),  # 1.9 (16 waves)
          ("f16", "nt", 2, 11008, 4096, "small"),  # 1.14 (rows)
          ("f16", "nt", 1, 16384, 2048, "small"),  # 1.3 (rows)
          ("f16", "nt", 1, 1024, 1024, "small"),  # 1.05 (rows)
          ("f32", "nt", 2, 32768, 2048, "small"),  # 1.25 with W from HBM (rows)
          ("f16", "nt", 32, 32768, 512, "tiles"),  # 1.33 (rows)
          ("f32", "nt", 64, 11008, 256, "tiles"),  # 1.17 (rows)
          ("f32", "nn", 64, 16384, 512, "tiles"),  # 1.16 (rows)
          ("f32", "nt", 64, 256, 8192, "tiles"),  # 1.35 (rows)
          ("f32", "nn", 64, 512, 2048, "small"),  # 1.29 (rows)
          ("f32", "nt", 16, 11008, 4096, "rows"), ("f16", "nn", 4, 11008, 4096, "rows"), ("f32", "nn", 64, 256, 4096, "rows"),
          ("f16", "nn", 64, 5000, 1024, "rows")]  # 1.3, 1.35, 1.5, 1.7 (small or tiles)


@pytest.mark.parametrize("dtype,layout,M,N,K,kernel", ROUTES)
def test_few_rows_take_the_kernel_that_measured_best(plan, dtype, layout, M, N, K, kernel):
    out = subprocess.run([plan, "route", dtype, layout, str(M), str(N), str(K)], capture_output=True, text=True).stdout
    assert out.strip() == kernel
