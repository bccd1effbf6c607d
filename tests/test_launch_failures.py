"""Launches that fail in the middle of a sequence (CPU only: the engine's host code on a fake HIP runtime).

The engine hands a failed launch to its caller as an error, and the caller may
go on.  What a sequence keeps on the device for its own later launches must not
pass for the next sequence's.
"""
import os
import re
import subprocess

import pytest

from streamgc_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))

DRIVER = r"""
#include <algorithm>
#include <cstdio>
#include <cstring>
#include "fake_hip.hpp"
#include "sgc_launch.hpp"
#include "streamgc.h"

static int fails = 0;
#define CHECK(c) do { if (!(c)) { std::printf("FAIL line %d: %s\n", __LINE__, #c); fails++; } } while (0)

static int at(const char* kernel, size_t from = 0) {   // the first launch of it, or -1
    for (size_t i = from; i < fake::launched.size(); i++)
        if (fake::launched[i].find(kernel) != std::string::npos) return (int)i;
    return -1;
}

constexpr uint32_t N = 64;
static std::vector<uint32_t> rp, col, deg;
static std::vector<sgc_edge_update> recs;

static sgc_engine* path_engine() {
    rp.assign(1, 0);
    col.clear();
    deg.clear();
    recs.clear();
    for (uint32_t v = 0; v < N; v++) {
        if (v) col.push_back(v - 1);
        if (v + 1 < N) col.push_back(v + 1);
        rp.push_back((uint32_t)col.size());
        deg.push_back(rp[v + 1] - rp[v]);
    }
    for (uint32_t v = 0; v + 1 < N; v++) {
        sgc_edge_update r;
        memset(&r, 0, sizeof r);
        r.u = v, r.v = v + 1, r.type = 1;
        recs.push_back(r);
    }
    sgc_config c;
    sgc_default_config(&c);
    c.flags |= SGC_REPAIR_EVERY_EPOCH;
    c.epoch_size = N;
    sgc_engine* e = nullptr;
    CHECK(sgc_create(&c, N, rp.data(), col.data(), deg.data(), &e) == SGC_OK);
    return e;
}

// A batch's edge table is emptied by the batch's own launches.
static void edge_table() {
    sgc_engine* e = path_engine();
    auto apply = [&] {
        fake::launched.clear();
        return sgc_apply(e, recs.data(), recs.size(), 0);
    };
    for (int k = 0; k < 2; k++) {
        CHECK(apply() == SGC_OK);
        CHECK(at("k_group_link") >= 0 && at("k_apply_") > at("k_group_pack") && at("k_group_clear") < 0);
    }
    for (const char* kernel : {"k_group_link", "k_group_pack", "k_apply_"}) {
        fake::fail_next = kernel;
        CHECK(apply() != SGC_OK && fake::fail_next.empty());
        CHECK(at("k_apply_") < 0);
        CHECK(apply() == SGC_OK);
        CHECK(at("k_group_clear") >= 0 && at("k_group_clear") < at("k_group_link"));
        CHECK(apply() == SGC_OK && at("k_group_clear") < 0);
    }
    sgc_destroy(e);
}

static uint32_t* control = nullptr;   // the control block of a batched run, on the "device"

// A captured round that stops for the host, its graph still iterating.
static void watch(void* dst, const void*, size_t bytes, int kind) {
    if (kind == (int)hipMemcpyHostToDevice && bytes == sgc::RC_WORDS * 4) control = (uint32_t*)dst;
    if (kind == (int)hipMemcpyDeviceToHost && bytes == sizeof(sgc::RoundState))
        *(sgc::RoundState*)dst = sgc::RoundState{1, 1000, 0, 2, 1000, 0};
}
static void stop() {
    control[sgc::RC_ROUND] = 0;
    control[sgc::RC_STOP] = 1;
    control[sgc::RC_STOP_ROUND] = 0;
}

// The worklist an epoch builds ahead, for the sweep after its drain, is that epoch's alone.
static void list_ahead() {
    sgc_engine* e = path_engine();
    sgc_batch_config c;
    sgc_default_batch_config(&c);
    uint32_t rounds = 0;
    for (bool failed : {false, true}) {
        CHECK(sgc_batch_prepare(e, recs.data(), recs.size(), &c, &rounds) == SGC_OK && rounds == 1);
        sgc_epoch_stats st;
        fake::launched.clear();
        if (failed) fake::fail_next = "k_drain";
        CHECK((sgc_epoch(e, &st) != SGC_OK) == failed && fake::fail_next.empty());
        CHECK((at("k_rebuild") < 0) == failed);
        CHECK((at("set") > at("k_list_tiles")) == failed);   // the listed vertices' marks are set again
        fake::on_copy = watch;
        fake::on_graph_launch = stop;
        fake::launched.clear();
        sgc_batch_stats bs;
        CHECK(sgc_batch_run(e, &bs) == SGC_OK && bs.host_rounds == 1);
        // the host's first sweep: the marked vertices are listed anew
        const int graph = at("graph"), sweep = std::min((unsigned)at("k_rebuild", graph), (unsigned)at("k_tier1", graph));
        CHECK(graph >= 0 && sweep > graph && at("k_list_tiles", graph) > graph && at("k_list_tiles", graph) < sweep);
        fake::on_copy = nullptr;
        fake::on_graph_launch = nullptr;
    }
    sgc_destroy(e);
}

int main() {
    edge_table();
    list_ahead();
    std::printf("%s\n", fails ? "FAILED" : "ok");
    return fails ? 1 : 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    """The driver, the engine's host code and the fake runtime in one program."""
    d = tmp_path_factory.mktemp("fake")
    (d / "driver.cpp").write_text(DRIVER)
    host = [build._hipcc(), *build.COMMON, "-O1", "-w", "-I", HERE]
    jobs, objs = [], []
    for src in [os.path.join(build.CSRC, s) for s in build.HIP_SOURCES]:
        objs.append(str(d / (os.path.basename(src) + ".o")))
        jobs.append([*host, f"--offload-arch={build.ARCH}", "--offload-host-only", "-c", src, "-o", objs[-1]])
    plain = [os.path.join(build.CSRC, "sgc_host.cpp"), os.path.join(HERE, "fake_hip.cpp"), str(d / "driver.cpp")]
    for src in plain:
        objs.append(str(d / (os.path.basename(src) + ".o")))
        jobs.append([*host, "-fopenmp", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-x", "c++", "-c", src, "-o",
                     objs[-1]])
    for p in [subprocess.Popen(j) for j in jobs]:
        assert p.wait() == 0
    # each host object refers to its device code's image by a name of its own
    names = subprocess.run(["nm", "-u", *objs], check=True, stdout=subprocess.PIPE, text=True).stdout
    images = sorted(set(re.findall(r"__hip_fatbin_\w+", names)))
    (d / "images.cpp").write_text("".join(f'extern "C" {{ char {n}[8]; }}\n' for n in images))
    exe = str(d / "program")
    subprocess.run(["g++", "-fopenmp", "-pthread", "-o", exe, *objs, str(d / "images.cpp")], check=True)
    return exe


def test_failed_launches_leave_nothing_behind(program):
    r = subprocess.run([program], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout + r.stderr
