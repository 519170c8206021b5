// Copies of a disk's fields to the host with pinned memory refused and granted,
// for tests/test_gpu_pinned.py: this program's hipHostMalloc stands before the
// runtime's, counts what the copies ask for and refuses it on request.
//
//   pinned_check <dir> [once]
// <dir> holds desc.bin (fcpt_disk_desc bytes, radii pointer ignored) and
// radii.bin.  Prints one line per copy: its name, "same" or "differ" (the copy
// without pinned memory against the one with it; "once", a process's first copy,
// against what was uploaded), the pinned allocations made and their bytes.
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/fcpt.h"

static bool refuse = false;
static size_t pins = 0, pinned_bytes = 0;

extern "C" hipError_t hipHostMalloc(void **p, size_t bytes, unsigned flags)
{
    using Fn = hipError_t (*)(void **, size_t, unsigned);
    static const Fn real = reinterpret_cast<Fn>(dlsym(RTLD_NEXT, "hipHostMalloc"));
    if (flags & hipHostMallocPortable) {  // the copies' staging; a context's own are not
        if (refuse) return hipErrorOutOfMemory;
        ++pins;
        pinned_bytes += bytes;
    }
    return real(p, bytes, flags);
}

static std::vector<char> slurp(const std::string &path)
{
    std::vector<char> b;
    if (FILE *f = std::fopen(path.c_str(), "rb")) {
        char t[4096];
        for (size_t n; (n = std::fread(t, 1, sizeof(t), f)) > 0;) b.insert(b.end(), t, t + n);
        std::fclose(f);
    }
    return b;
}

#define TRY(call)                                                                             \
    do {                                                                                      \
        if (const int rc = (call)) {                                                          \
            std::fprintf(stderr, "%s: %d %s\n", #call, rc, c ? fcpt_last_error(c) : "");      \
            return 1;                                                                         \
        }                                                                                     \
    } while (0)

int main(int argc, char **argv)
{
    if (argc < 2) return 2;
    const std::string dir = argv[1];
    const std::vector<char> db = slurp(dir + "/desc.bin"), rb = slurp(dir + "/radii.bin");
    fcpt_disk_desc desc;
    if (db.size() != sizeof(desc)) return 2;
    std::memcpy(&desc, db.data(), sizeof(desc));
    desc.radii = reinterpret_cast<const double *>(rb.data());
    fcpt_ctx *c = nullptr;
    TRY(fcpt_create(&desc, &c));
    const size_t rows[4] = {(size_t)desc.nr, (size_t)desc.nr + 1, (size_t)desc.nr, (size_t)desc.nr};
    std::vector<double> x[4], a[4], b[4];
    for (int f = 0; f < 4; ++f) {
        const size_t n = rows[f] * (size_t)desc.nphi;
        for (size_t k = 0; k < n; ++k) x[f].push_back(1.0 + 0.1 * std::sin(0.37 * (double)k + f));
        a[f].assign(n, 0.0);
        b[f].assign(n, -1.0);
    }
    TRY(fcpt_upload_state(c, x[0].data(), x[1].data(), x[2].data(), x[3].data()));
    auto state = [&](std::vector<double> *o) {
        return fcpt_download_state(c, o[0].data(), o[1].data(), o[2].data(), o[3].data());
    };
    auto report = [&](const char *name, int first, int last) {
        bool same = true;
        for (int f = first; f <= last; ++f)
            same = same && std::memcmp(a[f].data(), b[f].data(), a[f].size() * sizeof(double)) == 0;
        std::printf("%s %s %zu %zu\n", name, same ? "same" : "differ", pins, pinned_bytes);
        std::fflush(stdout);
    };
    if (argc > 2) {
        for (int f = 0; f < 4; ++f) a[f] = x[f];
        TRY(state(b));
        report("once", 0, 3);
        TRY(fcpt_destroy(c));
        return 0;
    }
    refuse = true;
    TRY(fcpt_download_field(c, FCPT_VRAD, a[1].data()));
    refuse = false;
    TRY(fcpt_download_field(c, FCPT_VRAD, b[1].data()));
    report("field", 1, 1);
    refuse = true;
    TRY(state(a));
    refuse = false;
    TRY(state(b));
    report("state", 0, 3);
    TRY(fcpt_destroy(c));
    return 0;
}
