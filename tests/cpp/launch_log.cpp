// What the library launches, on the host: the HIP runtime's entry points that it calls
// are defined here (they take precedence over libamdhip64's), memory is host memory,
// and a launch is printed instead of run:
//
//   [recorded ]name grid=G block=T[ order=bufK][ part=P][ out=bufK ...][ items=M]
//
// bufK is the K-th allocation.  A launch made while the stream is being captured is
// marked "recorded" and counts as not run; a read of an instance order that no launch
// that ran has written is marked "UNWRITTEN".
//
//   launch_log system n np tableau adaptive batch lanes ipw n_obs slots flags occ op...
//   op: solve forward adjoint:N sens observed capture end
#include <hip/hip_runtime_api.h>

#include <cxxabi.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <map>
#include <set>
#include <string>

#include "va_kernels.hpp"
#include "vectorizedadjoint_amd.h"

namespace {
std::map<const void *, std::string> &names()
{
    static std::map<const void *, std::string> m;
    return m;
}
std::map<char *, std::pair<size_t, int>> bufs;  // address -> size, number
std::set<const void *> written;                 // orders that a launch that ran has written
int n_bufs = 0, occupancy = 2;
size_t in_use = 0;  // bytes by hipMalloc
bool capturing = false, quiet = true;
struct Call {
    dim3 grid, block;
    size_t shmem;
    hipStream_t s;
} pending;

void *new_buf(size_t bytes)
{
    char *p = (char *)calloc(1, bytes + 64);
    bufs[p] = {bytes, n_bufs++};
    return p;
}
std::string buf(const void *p)
{
    if (!p) return "null";
    auto it = bufs.upper_bound((char *)p);
    if (it == bufs.begin()) return "?";
    --it;
    return (const char *)p < it->first + it->second.first ? "buf" + std::to_string(it->second.second)
                                                            : "?";
}
void order_read(const int32_t *order)
{
    printf(" order=%s%s", buf(order).c_str(),
           order && !capturing && !written.count(order) ? " UNWRITTEN" : "");
}
bool starts(const std::string &s, const char *p) { return s.compare(0, strlen(p), p) == 0; }

void log_launch(const void *f, dim3 g, dim3 b, void **args)
{
    auto it = names().find(f);
    std::string n = it == names().end() ? "?" : it->second;
    int st = 0;
    char *d = abi::__cxa_demangle(n.c_str(), nullptr, nullptr, &st);
    if (d) n = d;
    free(d);
    for (const char *drop : {"void ", "va::", "(anonymous namespace)::"})
        for (size_t k; (k = n.find(drop)) != std::string::npos;) n.erase(k, strlen(drop));
    n = n.substr(0, n.rfind('('));
    while (!n.empty() && n.back() == ' ') n.pop_back();
    if (starts(n, "k_iota_i32") && !capturing) written.insert(*(void **)args[0]);
    if (starts(n, "k_order_scatter") && !capturing) {
        const auto &a = *(const va::OrderArgs *)args[0];
        for (int m = 0; m < 2; ++m)
            if (a.modes >> m & 1) written.insert(a.order[m]);
    }
    if (quiet) return;
    printf("%s%s grid=%u block=%u", capturing ? "recorded " : "", n.c_str(), g.x, b.x);
    if (starts(n, "k_fwd") || (starts(n, "k_glv_rows") && n.find("_fwd") != std::string::npos)) {
        const auto &a = *(const va::FwdArgs *)args[0];
        order_read(a.order);
        printf(" part=%d", a.split ? a.part : -1);
    } else if (starts(n, "k_glv_rows_long<")) {
        order_read(((const va::FwdArgs *)args[0])->order);
    } else if (starts(n, "k_rev") || starts(n, "k_glv_rows")) {
        const auto &a = *(const va::RevArgs *)args[0];
        order_read(a.order);
        printf(" part=%d items=%d in_turn=%d", a.split ? a.part : -1, va::rev_items(a).parts,
               a.in_turn != nullptr);
    } else if (starts(n, "k_obs_fwd")) {
        order_read(((const va::ObsFwdArgs *)args[0])->order);
    } else if (starts(n, "k_obs_rev")) {
        order_read(((const va::ObsRevArgs *)args[0])->order);
    } else if (starts(n, "k_order_scatter")) {
        const auto &a = *(const va::OrderArgs *)args[0];
        if (a.from) order_read(a.from);
        for (int m = 0; m < 2; ++m)
            if (a.modes >> m & 1) printf(" out%d=%s long%d=%d", m, buf(a.order[m]).c_str(), m, a.long_bucket[m]);
    }
    printf("\n");
}
}  // namespace

extern "C" {
void **__hipRegisterFatBinary(const void *)
{
    static void *h;
    return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *,
                           void *, void *, void *, int *)
{
    names()[f] = name;
}
void __hipRegisterVar(void **, void *, char *, const char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, hipStream_t s)
{
    pending = {g, b, m, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *m, hipStream_t *s)
{
    *g = pending.grid, *b = pending.block, *m = pending.shmem, *s = pending.s;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t, hipStream_t)
{
    log_launch(f, g, b, args);
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int)
{
    *v = 256;
    return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetDevice(int *d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t)
{
    *n = occupancy;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n)
{
    const char *most = getenv("LAUNCH_LOG_MEMORY");  // bytes of the device; unset: any
    if (most && in_use + n > strtoull(most, nullptr, 10)) return hipErrorOutOfMemory;
    in_use += n;
    return *p = new_buf(n), hipSuccess;
}
hipError_t hipMallocAsync(void **p, size_t n, hipStream_t) { return *p = new_buf(n), hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return *p = new_buf(n), hipSuccess; }
hipError_t hipFree(void *p)
{
    if (p) in_use -= bufs[(char *)p].first;
    return hipSuccess;
}
hipError_t hipFreeAsync(void *, hipStream_t) { return hipSuccess; }
hipError_t hipHostFree(void *) { return hipSuccess; }
hipError_t hipMemset(void *, int, size_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t)
{
    return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void *, size_t, const void *, size_t, size_t, size_t, hipMemcpyKind,
                            hipStream_t)
{
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    return *s = (hipStream_t)new_buf(8), hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *st)
{
    *st = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode)
{
    capturing = true;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g)
{
    capturing = false;
    *g = (hipGraph_t)new_buf(8);
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t)
{
    return *e = (hipGraphExec_t)new_buf(8), hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t)
{
    printf("graph launch\n");
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return *e = (hipEvent_t)new_buf(8), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
}

int main(int argc, char **argv)
{
    if (argc < 13) return 2;
    va_problem pb;
    va_problem_init(&pb);
    int k = 1;
    auto num = [&]() { return atoi(argv[k++]); };
    pb.system = num();
    pb.n_state = num();
    pb.n_param = num();
    pb.tableau = num();
    pb.adaptive = num();
    pb.batch = num();
    pb.lanes = num();
    pb.instances_per_wave = num();
    pb.n_obs = num();
    pb.checkpoint_slots = num();
    pb.flags = num();
    occupancy = num();
    pb.t1 = 1.0;
    pb.dt0 = 1e-3;
    pb.abs_tol = pb.rel_tol = 1e-6;
    pb.max_steps = 8;
    va_handle *h = nullptr;
    auto check = [](va_status st) {
        if (st) {
            printf("error %d: %s\n", (int)st, va_last_error());
            exit(1);
        }
    };
    check(va_create(&pb, &h));
    quiet = false;
    double x[8] = {};  // stands for every array of the caller's: no launch reads it
    for (; k < argc; ++k) {
        const std::string op = argv[k];
        printf("-- %s\n", op.c_str());
        if (op == "capture") capturing = true;
        else if (op == "end") capturing = false;
        else if (op == "solve")
            check(va_solve(h, x, x, 1, nullptr, x, x, x, x, nullptr, nullptr, nullptr, nullptr));
        else if (op == "forward") check(va_forward(h, x, x, nullptr, nullptr, nullptr, nullptr));
        else if (starts(op, "adjoint:")) check(va_adjoint(h, x, atoi(op.c_str() + 8), x, x, nullptr));
        else if (op == "sens") check(va_sensitivity_matrix(h, x, x, nullptr));
        else if (op == "observed")
            check(va_solve_observed(h, x, x, x, x, x, x, x, x, nullptr, nullptr, nullptr, nullptr));
        else return 2;
    }
    return 0;
}
