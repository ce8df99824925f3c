// Runs k_run_order (pyjess_amd/csrc/jam_ingest.h) on the CPU under the HIP
// emulation of hip/hip_runtime.h, over the last atoms of a batch as large as one may
// be: two small molecules whose serial numbers descend at a few atoms, behind one
// of BEFORE atoms that nothing reads. Test infrastructure only.
//
//   order_emu BEFORE
// Exits with 1 where the order is not that of a stable sort.

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <numeric>
#include <vector>

#include <sys/mman.h>

#include <hip/hip_runtime.h>

struct uint4 {
    unsigned x, y, z, w;
};

#define __constant__ const

#include "jam_ingest.h"

using namespace jam;

static unsigned first_block;

static void run_order(const int *atom_off, int n_mols, const int *serial, const int *down, int n_down, int *order)
{
    emu::t_block.x += first_block;
    k_run_order(atom_off, n_mols, serial, down, n_down, order);
}

// n zeros, of which only what is touched takes memory
static int *sparse(size_t n)
{
    void *p = mmap(nullptr, n * sizeof(int), PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (p == MAP_FAILED) {
        std::perror("mmap");
        std::exit(2);
    }
    return (int *)p;
}

int main(int argc, char **argv)
{
    const int before = argc > 1 ? std::atoi(argv[1]) : 0, sizes[2] = {700, 300};
    const std::vector<int> atom_off = {0, before, before + sizes[0], before + sizes[0] + sizes[1]};
    const size_t na = (size_t)atom_off[3];
    int *serial = sparse(na), *order = sparse(na);
    std::vector<int> down;
    for (int m = 1; m <= 2; m++)
        for (int a = atom_off[m]; a < atom_off[m + 1]; a++) {
            serial[a] = (a - atom_off[m]) % (m == 1 ? 190 : 299) / 2;
            if (a > atom_off[m] && serial[a] < serial[a - 1]) down.push_back(a);
        }
    first_block = (unsigned)(before / ING_THREADS);
    const unsigned last_block = (unsigned)((na - 1) / ING_THREADS);
    // (atoms of the large molecule that share the first block are ranked in a run of their own, not read)
    emu::launch(run_order, dim3(last_block - first_block + 1), dim3(ING_THREADS), (const int *)atom_off.data(), 3,
                (const int *)serial, (const int *)down.data(), (int)down.size(), order);
    for (int m = 1; m <= 2; m++) {
        std::vector<int> want(sizes[m - 1]);
        std::iota(want.begin(), want.end(), 0);
        const int *sr = serial + atom_off[m];
        std::stable_sort(want.begin(), want.end(), [sr](int x, int y) { return sr[x] < sr[y]; });
        if (!std::equal(want.begin(), want.end(), order + atom_off[m])) {
            std::printf("molecule %d: wrong order\n", m);
            return 1;
        }
    }
    std::printf("%zu descents\n", down.size());
    return 0;
}
