"""The global loads and stores of the FP32 ring and narrow GEMM bodies, without
a GPU: the headers compiled as host C++, every lane of every block run at sizes
whose last tiles, K steps and K ranges are cut short. A buffer access must have
offsets at or past its base (they are unsigned on the device) and lie inside its
operand; plain accesses are caught by inaccessible pages right before and right
after each operand."""

import subprocess
from pathlib import Path

import pytest

CLANG = "/opt/rocm/llvm/bin/clang++"
HIP = Path(__file__).resolve().parent.parent / "minicompiler_amd" / "csrc" / "hip"

SHIM = r"""
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <initializer_list>
#include <sys/mman.h>
#include <unistd.h>
struct Dim { unsigned x; };
static Dim threadIdx, blockIdx, gridDim;
struct Rsrc { char* base; };
static char *lo[3], *hi[3];  // A, B, C
static const char* now = "";
static char* checked(Rsrc r, int voffset, int soffset, int bytes) {
    char* p = r.base + voffset + soffset;
    bool inside = false;
    for (int i = 0; i < 3; ++i) inside = inside || (p >= lo[i] && p + bytes <= hi[i]);
    if (voffset >= 0 && soffset >= 0 && inside) return p;
    std::printf("%s: block %u lane %u: offsets %d + %d (%s)\n", now, blockIdx.x, threadIdx.x, voffset, soffset,
                inside ? "before the base" : "outside the operands");
    std::exit(1);
}
template <typename T> static T load(Rsrc r, int v, int s) { T t; std::memcpy(&t, checked(r, v, s, sizeof(T)), sizeof(T)); return t; }
template <typename T> static void store(T t, Rsrc r, int v, int s) { std::memcpy(checked(r, v, s, sizeof(T)), &t, sizeof(T)); }
typedef unsigned U2 __attribute__((ext_vector_type(2)));
typedef unsigned U4 __attribute__((ext_vector_type(4)));
#define __device__
#define __forceinline__ inline
#define __shared__ static
#define __syncthreads()
#define __amdgpu_buffer_rsrc_t Rsrc
#define __builtin_amdgcn_make_buffer_rsrc(p, stride, n, flags) Rsrc{(char*)(p)}
#define __builtin_amdgcn_raw_buffer_load_b128(r, v, s, x) load<U4>(r, v, s)
#define __builtin_amdgcn_raw_buffer_load_b64(r, v, s, x) load<U2>(r, v, s)
#define __builtin_amdgcn_raw_buffer_load_b32(r, v, s, x) load<unsigned>(r, v, s)
#define __builtin_amdgcn_raw_buffer_store_b128(t, r, v, s, x) store(t, r, v, s)
#define __builtin_amdgcn_raw_buffer_store_b64(t, r, v, s, x) store(t, r, v, s)
#define __builtin_amdgcn_raw_buffer_store_b32(t, r, v, s, x) store(t, r, v, s)
#define __builtin_amdgcn_raw_ptr_buffer_load_lds(r, dst, bytes, v, s, o, x) (void)checked(r, v, s, bytes)
#define __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, x, y, z) (c)
#define __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, x, y, z) (c)
#define __builtin_amdgcn_readfirstlane(x) (x)
#define __builtin_amdgcn_sched_barrier(x)
#define __builtin_amdgcn_sched_group_barrier(x, y, z)
#define __builtin_amdgcn_s_waitcnt(x)
#define __builtin_amdgcn_s_barrier()
#define __HIP_MEMORY_SCOPE_AGENT 0
#define __hip_atomic_store(p, v, o, s) (void)(*(p) = (v))
#define __hip_atomic_load(p, o, s) (*(p))
#define __hip_atomic_fetch_add(p, v, o, s) ((*(p) += (v)) - (v))
"""

MAIN = r"""
struct Store { float operator()(float v, unsigned) const { return v; } };

// A buffer of `count` floats that starts (or ends) at an inaccessible page.
struct Guarded {
    char* map; size_t pages, page = sysconf(_SC_PAGESIZE); float* p;
    Guarded(size_t count, bool at_end) {
        pages = (4 * count + page - 1) / page;
        map = (char*)mmap(nullptr, (pages + 2) * page, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
        mprotect(map + page, pages * page, PROT_READ | PROT_WRITE);
        p = (float*)(map + page + (at_end ? pages * page - 4 * count : 0));
    }
    ~Guarded() { munmap(map, (pages + 2) * page); }
};

template <class Run>
static void blocks(const char* name, int m, int n, int k, int k_split, int tiles, int threads, const Run& run) {
    const int depth = (k + k_split - 1) / k_split;
    char text[160];
    std::snprintf(text, sizeof text, "%s %dx%dx%d in %d of %d", name, m, n, k, depth, k_split);
    now = text;
    std::printf("%s\n", text);
    for (bool at_end : {false, true}) {
        Guarded a((size_t)m * k, at_end), b((size_t)k * n, at_end), c((size_t)m * n * depth, at_end);
        Guarded* g[3] = {&a, &b, &c};
        const size_t count[3] = {(size_t)m * k, (size_t)k * n, (size_t)m * n * depth};
        for (int i = 0; i < 3; ++i) lo[i] = (char*)g[i]->p, hi[i] = lo[i] + 4 * count[i];
        gridDim.x = (unsigned)(tiles * depth);
        for (blockIdx.x = 0; blockIdx.x < gridDim.x; ++blockIdx.x)
            for (threadIdx.x = 0; threadIdx.x < (unsigned)threads; ++threadIdx.x) run(a.p, b.p, c.p, depth);
    }
}

static int up(int a, int b) { return (a + b - 1) / b; }

template <class Cfg, bool kRagged>
static void narrow(const char* name, int m, int n, int k, int k_split) {
    blocks(name, m, n, k, k_split, up(m, Cfg::kRows) * up(n, Cfg::kCols), Cfg::kThreads,
           [&](float* a, float* b, float* c, int depth) {
               mc_gemm_f32_narrow<Cfg, kRagged>(a, b, c, m, n, k, k_split, depth, depth > 1 ? c : nullptr, nullptr, Store{});
           });
}

template <class Cfg, bool kRagged>
static void ring(const char* name, int m, int n, int k, int k_split) {
    blocks(name, m, n, k, k_split, up(m, Cfg::kBM) * up(n, Cfg::kBN), Cfg::kThreads,
           [&](float* a, float* b, float* c, int depth) {
               mc_gemm_f32_ring<Cfg, kRagged>(a, b, c, m, n, k, k_split, depth, depth > 1 ? c : nullptr, nullptr, Store{});
           });
}

template <class Cfg>
static void narrow_sizes(const char* name) {
    constexpr int R = Cfg::kRows, C = Cfg::kCols;
    for (int n : {C + 1, C + 2, C + 3, 2 * C - 1, C, C + 4, 4, 6})
        for (int k : {16, 17, 31, 33, 100}) narrow<Cfg, true>(name, Cfg::kStreamB ? R : R + 1, n, k, 16 * up(k, 16));
    narrow<Cfg, true>(name, R, C + 1, 200, 64);
    narrow<Cfg, true>(name, 1, C + 1, 129, 64);
    narrow<Cfg, false>(name, R - 1, C + 4, 96, 96);
    narrow<Cfg, false>(name, R, 2 * C, 160, 64);
}

template <class Cfg>
static void ring_sizes(const char* name, bool ragged) {
    if constexpr (Cfg::kStaged && Cfg::kStages == 2 && Cfg::kBM == 128) {
        if (ragged) {
            for (int n : {129, 130, 131, 4, 132})
                for (int k : {64, 65, 95, 97}) ring<Cfg, true>(name, 129, n, k, 32 * up(k, 32));
            ring<Cfg, true>(name, 130, 257, 129, 64);
        }
    }
    ring<Cfg, false>(name, Cfg::kBM + 1, Cfg::kBN + 4, 96, 96);
    ring<Cfg, false>(name, 1, 4, 160, 64);
}

int main(int, char** argv) {
    const char* what = argv[1];
    if (!std::strcmp(what, "narrow")) {
        narrow_sizes<McNarrow16>("16x64 streamed");
        narrow_sizes<McNarrow32>("32x64");
        narrow_sizes<McNarrow16x64>("16x64");
        narrow_sizes<McNarrow16x32>("16x32");
        narrow_sizes<McNarrow16x32Sums>("16x32 with more sums");
        narrow_sizes<McNarrow64>("64x64");
        narrow_sizes<McNarrow16x16>("16x16");
    } else {
        ring_sizes<McRingWide>("wide", true);
        ring_sizes<McRingWide8>("wide8", true);
        ring_sizes<McRingMid>("mid", false);
        ring_sizes<McRingBig>("big", false);
        ring_sizes<McRingThin>("thin", false);
    }
    std::puts("ok");
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("offsets")
    text = "".join((HIP / h).read_text().replace("#pragma once", "")
                   for h in ("gemm_split_arrival.h", "gemm_f32_ring.h", "gemm_f32_narrow.h"))
    text = text.replace("__attribute__((address_space(3)))", "").replace("#pragma unroll", "")
    (tmp / "offsets.cpp").write_text(SHIM + text + MAIN)
    subprocess.run([CLANG, "-std=c++20", "-O1", "-w", str(tmp / "offsets.cpp"), "-o", str(tmp / "offsets")], check=True)
    return tmp / "offsets"


@pytest.mark.parametrize("body", ["narrow", "ring"])
def test_every_access_is_at_or_past_its_base_and_inside_its_operand(program, body):
    run = subprocess.run([str(program), body], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0 and run.stdout.endswith("ok\n"), (run.returncode, run.stdout[-300:], run.stderr[-300:])
