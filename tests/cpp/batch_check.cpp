// Host waits of fcpt_batch_run_steps, for tests/test_gpu_batch_own_fields.py: this
// program's hipStreamSynchronize stands before the runtime's and counts.
//
//   batch_check <dir> <members>
// <dir> holds desc.bin (fcpt_disk_desc bytes, radii pointer ignored), radii.bin,
// sigma.bin, vrad.bin, vazi.bin and energy.bin.  Prints the waits of two steps of
// the batch as it is, after its first member's pressure has been uploaded, and
// after that member has stepped alone.
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/fcpt.h"

static int waits = 0;

extern "C" hipError_t hipStreamSynchronize(hipStream_t s)
{
    using Fn = hipError_t (*)(hipStream_t);
    static const Fn real = reinterpret_cast<Fn>(dlsym(RTLD_NEXT, "hipStreamSynchronize"));
    ++waits;
    return real(s);
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
            std::fprintf(stderr, "%s: %d\n", #call, rc);                                      \
            return 1;                                                                         \
        }                                                                                     \
    } while (0)

int main(int argc, char **argv)
{
    if (argc < 3) return 2;
    const std::string dir = argv[1];
    const std::vector<char> db = slurp(dir + "/desc.bin"), rb = slurp(dir + "/radii.bin");
    fcpt_disk_desc desc;
    if (db.size() != sizeof(desc)) return 2;
    std::memcpy(&desc, db.data(), sizeof(desc));
    desc.radii = reinterpret_cast<const double *>(rb.data());
    std::vector<char> x[4];
    const char *names[4] = {"/sigma.bin", "/vrad.bin", "/vazi.bin", "/energy.bin"};
    for (int f = 0; f < 4; ++f) x[f] = slurp(dir + names[f]);
    auto p = [&](int f) { return reinterpret_cast<const double *>(x[f].data()); };
    std::vector<fcpt_ctx *> disks((size_t)std::atoi(argv[2]));
    for (fcpt_ctx *&c : disks) {
        TRY(fcpt_create(&desc, &c));
        TRY(fcpt_upload_reference(c, p(0), p(1), p(2), p(3)));
        TRY(fcpt_upload_state(c, p(0), p(1), p(2), p(3)));
        TRY(fcpt_set_time(c, 0.0, 0.1, 0));
    }
    fcpt_batch *b = nullptr;
    TRY(fcpt_batch_create(disks.data(), (int)disks.size(), &b));
    TRY(fcpt_batch_run_steps(b, 2, 1));
    std::vector<double> pr((size_t)desc.nr * (size_t)desc.nphi);
    for (int how = 0; how < 3; ++how) {
        if (how == 1) {
            TRY(fcpt_download_field(disks[0], FCPT_PRESSURE, pr.data()));
            TRY(fcpt_upload_field(disks[0], FCPT_PRESSURE, pr.data()));
        }
        if (how == 2) TRY(fcpt_run_steps(disks[0], 1, 0));
        waits = 0;
        TRY(fcpt_batch_run_steps(b, 2, 1));
        std::printf("%d\n", waits);
    }
    TRY(fcpt_batch_synchronize(b));
    TRY(fcpt_batch_destroy(b));
    for (fcpt_ctx *c : disks) TRY(fcpt_destroy(c));
    return 0;
}
