"""The upload of the J/K tile lists (gtfock_amd/csrc/engine.cpp), built for the
host with stand-ins for the device: the gathered copy, and what is left of the
classes' tiles when an allocation fails."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gtfock_amd", "csrc")

SRC = r"""
#include "eri_kernels.h"
#include "engine.h"
#include "screen.h"
#include <cstring>

static int fail_in = -1;  // allocations until one fails
extern "C" {
hipError_t hipMalloc(void** p, size_t n)
{
    *p = fail_in >= 0 && fail_in-- == 0 ? nullptr : malloc(n);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { memset(d, v, n); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamCreate(hipStream_t*) { return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t*) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t*, unsigned) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float*, hipEvent_t, hipEvent_t) { return hipSuccess; }
hipError_t hipGetDevice(int*) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int*, hipDeviceAttribute_t, int) { return hipSuccess; }
hipError_t hipFuncGetAttributes(hipFuncAttributes*, const void*) { return hipErrorUnknown; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return ""; }
}
int gtf_jk_begin(hipStream_t, const JkLists&, const double*, double*, double*, long, int, long, int*, int) { return 0; }
int gtf_jk_end(hipStream_t, const JkLists&, double*, int, long) { return 0; }
int gtf_fill_int(hipStream_t, int*, long, int) { return 0; }
int gtf_round_f32(hipStream_t, const double*, long, float*) { return 0; }
int gtf_pack_kets(hipStream_t, const PairView&, const int*, const KetPack&) { return 0; }
int gtf_build_pairs(hipStream_t, const BasisView&, int, const int*, const int*, const int*, const long*, double4*, double*,
                    const long*, double*, int*, double*, double) { return 0; }
int gtf_prim_census(hipStream_t, const CensusArgs&) { return 0; }
size_t gtf_sig_temp_bytes(int) { return 0; }
int gtf_fill_qlist_diag(hipStream_t, int, const int*, int2*) { return 0; }
int gtf_symmetrize_packed(hipStream_t, double*, int, const long*, const int*, int) { return 0; }
int gtf_sig_count(hipStream_t, int, const int*, int, const unsigned long long*, const int*, const double*, int*, int*, int*) { return 0; }
int gtf_sig_order(hipStream_t, int, const int*, int, const unsigned long long*, const int*, const double*, const int*, int,
                  const int*, int, SigWork&, SigOut&) { return 0; }
int gtf_count_rows(hipStream_t, int, const int*, const int*, const double*, const int*, const double*, const int*, const int*,
                   const int*, double, int, long*, long*, long*) { return 0; }
const EriClassInfo* gtf_eri_class(int) { static const EriClassInfo e{}; return &e; }
void gtf_boys_table(double*, int, int, double) {}
void gtf_boys_taylor_tables(double*) {}

static GtfSystem::TileList make(int c, int low, long n)
{
    GtfSystem::TileList t;
    for (long k = 0; k < n; k++) {
        TileHead h{};
        h.row = (int)k;
        h.bra = c;
        h.nrun = low;
        t.tiles.push_back(h);
        t.runs.push_back(make_int4((int)k, c, low, 7));
        t.runs.push_back(make_int4((int)k, c, low, 9));
    }
    return t;
}

static bool holds(const GtfSystem& s, int c, const GtfSystem::TileList& hv, const GtfSystem::TileList& lv)
{
    return s.nruns[c] == (int)hv.runs.size() && s.nruns_lo[c] == (int)lv.runs.size() &&
           !memcmp(s.d_tiles[c], hv.tiles.data(), hv.tiles.size() * sizeof(TileHead)) &&
           !memcmp(s.d_tiles_lo[c], lv.tiles.data(), lv.tiles.size() * sizeof(TileHead)) &&
           !memcmp(s.d_runs[c], hv.runs.data(), hv.runs.size() * sizeof(int4)) &&
           !memcmp(s.d_runs_lo[c], lv.runs.data(), lv.runs.size() * sizeof(int4));
}

static bool empty(const GtfSystem& s, int c)
{
    return !s.ntiles[c] && !s.ntiles_lo[c] && !s.nruns[c] && !s.nruns_lo[c] && !s.d_tiles[c] && !s.d_tiles_lo[c] &&
           !s.d_runs[c] && !s.d_runs_lo[c] && !s.tile_mem[c] && !s.nq_lo[c];
}

#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)

int main()
{
    GtfSystem s;
    GtfSystem::TileList hv[GTF_NCLASSES], lv[GTF_NCLASSES];
    // none, a few, and lists over several of the 4 MB pieces
    for (int c = 0; c < GTF_NCLASSES; c++) {
        hv[c] = make(c, 0, c == 3 ? 150000 : c % 4 ? 5 * c : 0);
        lv[c] = make(c, 1, c == 7 ? 70001 : c % 3);
    }
    auto count = [&]() {
        for (int c = 0; c < GTF_NCLASSES; c++) {
            s.ntiles[c] = (int)hv[c].tiles.size();
            s.ntiles_lo[c] = (int)lv[c].tiles.size();
            s.nq_lo[c] = s.ntiles_lo[c];
        }
    };
    count();
    CHECK(s.upload_tiles(hv, lv, 0, GTF_NCLASSES) == 0);
    for (int c = 0; c < GTF_NCLASSES; c++) CHECK(holds(s, c, hv[c], lv[c]));
    // one class alone: the others keep the shared allocation
    hv[5] = make(5, 0, 11);
    count();
    CHECK(s.upload_tiles(hv, lv, 5, 6) == 0);
    for (int c = 0; c < GTF_NCLASSES; c++) CHECK(holds(s, c, hv[c], lv[c]));
    // an allocation that fails leaves a class without tiles, the others as they were
    fail_in = 0;
    CHECK(s.upload_tiles(hv, lv, 5, 6) == -1);
    for (int c = 0; c < GTF_NCLASSES; c++) CHECK(c == 5 ? empty(s, c) : holds(s, c, hv[c], lv[c]));
    fail_in = 0;
    CHECK(s.upload_tiles(hv, lv, 0, GTF_NCLASSES) == -1);
    for (int c = 0; c < GTF_NCLASSES; c++) CHECK(empty(s, c));
    count();
    CHECK(s.upload_tiles(hv, lv, 0, GTF_NCLASSES) == 0);
    for (int c = 0; c < GTF_NCLASSES; c++) CHECK(holds(s, c, hv[c], lv[c]));
    printf("ok\n");
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="no hipcc")
def test_tile_upload(tmp_path):
    (tmp_path / "t.cpp").write_text(SRC)
    objs = []
    for src in (os.path.join(CSRC, "engine.cpp"), str(tmp_path / "t.cpp")):
        objs.append(str(tmp_path / (os.path.basename(src) + ".o")))
        subprocess.check_call(["hipcc", "--cuda-host-only", "-x", "hip", "--offload-arch=gfx950", "-O1", "-std=c++17", "-w",
                               "-I", CSRC, "-c", src, "-o", objs[-1]])
    exe = str(tmp_path / "t")
    subprocess.check_call(["g++", "-no-pie", "-o", exe] + objs + ["-lpthread"])
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr
