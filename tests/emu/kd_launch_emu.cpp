// Runs the kd kernels (pyjess_amd/csrc/jam_kd.h) on the CPU under the HIP
// emulation of hip/hip_runtime.h, through the library's own list of launches
// (kd_launches), so that the kernels, their launch shapes and their order are
// those of the device. Test infrastructure only.
//
//   kd_launch_emu INPUT OUTPUT
// INPUT: int32 n_sets, int32 one_molecule, int64 off[n_sets + 1],
//        double xyz[3 * off[n_sets]]
// OUTPUT: int32 order[off[n_sets]] -- per set, its points in leaf order
//         (left subtree first), set-local indices -- then int32 kd_err.
// Prints a line per launch: stream, slot among the grids (-1: none), threads.
// Side streams run in launch order, which is one of the orders that a device
// may take. Buffers that the kernels write before they read are filled with
// 0xFF bytes first.

#include <cstdio>
#include <cstring>
#include <vector>

#include "jam_kd.h"

using namespace jam;

template <class T>
static T *poisoned(std::vector<T> &v, size_t n)
{
    v.resize(n ? n : 1);
    std::memset((void *)v.data(), 0xFF, sizeof(T) * v.size());
    return v.data();
}

struct EmuQueue {
    unsigned open = 0, joined_ = 0;   // side streams

    template <class... K, class... A>
    void run(int k, int slot, void (*kernel)(K...), int threads, A... args)
    {
        std::printf("%d %d %d\n", k, slot, threads);
        launch(k, 2, kernel, threads, args...);   // a small grid: the kernels stride over their sets
    }
    template <class... K, class... A>
    void run_grid(int k, int blocks, void (*kernel)(K...), int threads, A... args)
    {
        std::printf("%d -1 %d\n", k, threads);
        launch(k, blocks, kernel, threads, args...);
    }
    template <class... K, class... A>
    void launch(int k, int blocks, void (*kernel)(K...), int threads, A... args)
    {
        // a side stream is forked before it is used, and joined after
        if (k != KD_MAIN && (!((open >> k) & 1u) || ((joined_ >> k) & 1u))) std::abort();
        emu::launch(kernel, dim3((unsigned)blocks), dim3((unsigned)threads), args...);
    }
    void fork(int k, int from)
    {
        if (k != from && !((open >> from) & 1u)) std::abort();
        open |= 1u << k;
    }
    void joined(int k) { joined_ |= 1u << k; }
};

int main(int argc, char **argv)
{
    if (argc != 3) {
        std::fprintf(stderr, "usage: kd_launch_emu INPUT OUTPUT\n");
        return 2;
    }
    FILE *f = std::fopen(argv[1], "rb");
    if (!f) return 2;
    int32_t n_sets = 0, one_molecule = 0;
    if (std::fread(&n_sets, 4, 1, f) != 1 || std::fread(&one_molecule, 4, 1, f) != 1) return 2;
    std::vector<int64_t> off(n_sets + 1);
    if (std::fread(off.data(), 8, off.size(), f) != off.size()) return 2;
    const int64_t total = off[n_sets];
    std::vector<double> xyz(3 * (size_t)total);
    if (std::fread(xyz.data(), 8, xyz.size(), f) != xyz.size()) return 2;
    std::fclose(f);

    // set s is molecule s with one atom type, its list its atoms in input order
    std::vector<int> atom_off(off.begin(), off.end()), chain(total, 0), resseq(total, 0), cnt(n_sets), list(total);
    int maxcnt = 0;
    for (int s = 0; s < n_sets; s++) {
        cnt[s] = (int)(off[s + 1] - off[s]);
        maxcnt = std::max(maxcnt, cnt[s]);
        for (int e = 0; e < cnt[s]; e++) list[off[s] + e] = e;
    }
    DevMols ms{};
    ms.n_mols = n_sets;
    ms.atom_off = atom_off.data();
    ms.xyz = xyz.data();
    ms.chain = chain.data();
    ms.resseq = resseq.data();
    DevTpls tp{};
    tp.n_types = 1;
    std::vector<int> kidx, l2k, katom, bucket, tied;
    std::vector<SetEnt> kent;
    std::vector<double> bbox, sbox;
    std::vector<unsigned char> scr;
    std::vector<unsigned int> count;
    int64_t total_dev = total;
    unsigned int kd_err = 0;
    DevSets st{};
    st.n_sets = n_sets;
    st.cap = total;
    st.blk_cap = total / JAM_WAVE + n_sets + 1;
    st.cnt = cnt.data();
    st.off = off.data();
    st.list = list.data();
    st.kidx = poisoned(kidx, total);
    st.l2k = poisoned(l2k, total);
    st.kent = poisoned(kent, total);
    st.katom = poisoned(katom, total);
    st.bbox = poisoned(bbox, 6 * (size_t)st.blk_cap);
    st.sbox = poisoned(sbox, 6 * (size_t)(total / JAM_SUB + n_sets + 1));
    st.total = &total_dev;
    st.maxcnt = &maxcnt;
    st.kd_err = &kd_err;
    EmuQueue q;
    kd_launches(q, ms, tp, st, poisoned(scr, (size_t)KD_SCRATCH_BYTES_PER_ENTRY * total),
                poisoned(bucket, (size_t)KD_TIERS * n_sets), poisoned(tied, (size_t)KD_TIERS * n_sets),
                poisoned(count, 2 * KD_TIERS), one_molecule != 0, total);
    if (q.open != q.joined_) std::abort();

    // kd DFS position p (right child first) holds list element kidx[p] and is
    // leaf n - 1 - p
    std::vector<int32_t> order(total);
    for (int s = 0; s < n_sets; s++)
        for (int j = 0; j < cnt[s]; j++) order[off[s] + j] = kidx[off[s] + cnt[s] - 1 - j];
    FILE *o = std::fopen(argv[2], "wb");
    if (!o) return 2;
    std::fwrite(order.data(), 4, (size_t)total, o);
    const int32_t err = (int32_t)kd_err;
    std::fwrite(&err, 4, 1, o);
    std::fclose(o);
    return 0;
}
