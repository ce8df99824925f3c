// Runs the kernels that order complete matches by groups of level-0 rows
// (k_group_* in pyjess_amd/csrc/jam_kernels.h) on the CPU under the HIP emulation
// of hip/hip_runtime.h, over made-up matches, and compares their order with a
// comparison sort's. Test infrastructure only.
//
//   sort_emu SEED MOLECULES ENTRIES ROWS MATCHES SHIFT WAY SIZE...
// SIZE...: atoms of each template; ENTRIES: most entries of a candidate set; up
// to MATCHES matches to each of ROWS level-0 rows; SHIFT: bits by which the row
// numbers are shortened; WAY: "ranked" (every group) or "tiled" (in LDS, larger
// groups listed and ranked). Prints: matches, largest group, key words, matches
// that share their first key word with another of their group; exits with 1
// where the order is wrong. Buffers are filled with 0xFF bytes first.

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <numeric>
#include <random>
#include <set>
#include <string>
#include <vector>

#include <hip/hip_runtime.h>

// what the kernels use beyond the emulation's header
struct int4 {
    int x, y, z, w;
};
struct double2 {
    double x, y;
};
inline int4 make_int4(int a, int b, int c, int d) { return {a, b, c, d}; }
inline int __clz(int v) { return v == 0 ? 32 : __builtin_clz((unsigned)v); }
inline float __double2float_ru(double d)
{
    const float f = (float)d;
    return (double)f < d ? std::nextafterf(f, INFINITY) : f;
}
template <class To, class From>
inline To as_bits(From v)
{
    To r;
    static_assert(sizeof(r) == sizeof(v), "");
    std::memcpy(&r, &v, sizeof(r));
    return r;
}
inline float __int_as_float(int i) { return as_bits<float>(i); }
inline int __float_as_int(float f) { return as_bits<int>(f); }

#include "jam_kernels.h"

using namespace jam;

template <class T>
static T *poisoned(std::vector<T> &v, size_t n)
{
    v.resize(n ? n : 1);
    std::memset((void *)v.data(), 0xFF, sizeof(T) * v.size());
    return v.data();
}

int main(int argc, char **argv)
{
    if (argc < 9) return 2;
    std::mt19937 rng((unsigned)std::atoi(argv[1]));
    const int M = std::atoi(argv[2]), entries = std::atoi(argv[3]), rows = std::atoi(argv[4]);
    const int per_row = std::atoi(argv[5]), shift = std::atoi(argv[6]);
    const bool rank_all = std::string(argv[7]) == "ranked";
    std::vector<int> size;
    for (int k = 8; k < argc; k++) size.push_back(std::atoi(argv[k]));
    const int T = (int)size.size(), P = M * T, stride = *std::max_element(size.begin(), size.end());

    // a set per pair and level, its kd positions in some list order
    std::vector<int> atom_off(T + 1, 0), kidx, nchunk(P), n1(P);
    std::vector<long long> base(P + 1, 0);
    std::vector<PairLevel> lvl((size_t)P * JAM_MAX_LEVELS);
    for (int t = 0; t < T; t++) atom_off[t + 1] = atom_off[t] + size[t];
    int maxcnt = 0;
    for (int p = 0; p < P; p++) {
        for (int l = 0; l < size[p % T]; l++) {
            const int c = 1 + (int)(rng() % entries);
            PairLevel &h = lvl[(size_t)p * JAM_MAX_LEVELS + l];
            h = PairLevel{};
            h.cnt = c;
            h.off = (int)kidx.size();
            std::vector<int> order(c);
            std::iota(order.begin(), order.end(), 0);
            std::shuffle(order.begin(), order.end(), rng);
            kidx.insert(kidx.end(), order.begin(), order.end());
            maxcnt = std::max(maxcnt, c);
        }
        n1[p] = size[p % T] == 1;
        nchunk[p] = lvl[(size_t)p * JAM_MAX_LEVELS].cnt - n1[p];
        base[p + 1] = base[p] + nchunk[p];
    }
    // matches: some rows, two choices at most levels, so that keys begin alike
    std::set<std::vector<int>> seen;   // pair, then an entry per level
    for (int r = 0; r < rows; r++) {
        const int p = (int)(rng() % P), n = size[p % T];
        const PairLevel *lv = &lvl[(size_t)p * JAM_MAX_LEVELS];
        const int e0 = lv[0].off + (int)(rng() % lv[0].cnt);
        if (n1[p] && kidx[e0] == 0) continue;   // a one-atom template steps past list entry 0
        for (int q = 0; q < per_row; q++) {
            std::vector<int> v{p, e0};
            for (int l = 1; l < n; l++)
                v.push_back(lv[l].off + (int)(rng() % (rng() % 8 ? std::min(lv[l].cnt, 2) : lv[l].cnt)));
            seen.insert(v);
        }
    }
    std::vector<std::vector<int>> match(seen.begin(), seen.end());
    std::shuffle(match.begin(), match.end(), rng);
    const long long n = (long long)match.size();
    if (n == 0) return 2;
    std::vector<int> pair, ent;
    for (auto &v : match) {
        pair.push_back(v[0]);
        for (int l = 0; l < stride; l++) ent.push_back(l + 1 < (int)v.size() ? v[l + 1] : -7);
    }
    DevTpls tp{};
    tp.n_templates = T;
    tp.atom_off = atom_off.data();
    DevSets st{};
    st.kidx = kidx.data();
    DevPairs pr{};
    pr.n_pairs = P;
    pr.lvl = lvl.data();
    pr.nchunk = nchunk.data();
    pr.n1 = n1.data();
    pr.item_base = base.data();
    DevJoin jn{};
    jn.stride = stride;
    jn.done_pair = pair.data();
    jn.done_ent = ent.data();

    // as the library launches them
    const int half = GROUP_TILE / 2, least = rank_all ? 1 : half + 1;
    const long long groups = (base[P] >> shift) + 1;
    std::vector<unsigned int> row;
    std::vector<int> slot, perm, list, count(groups, 0), start(groups + 1, 0), pos[2];
    std::vector<unsigned long long> key[2], work(4, 0);
    std::vector<GroupSeg> seg[2];
    poisoned(row, n);
    poisoned(slot, n);
    poisoned(perm, n);
    poisoned(list, n);
    for (int k = 0; k < 2; k++) {
        poisoned(pos[k], n);
        poisoned(key[k], n);
        poisoned(seg[k], n);
    }
    const unsigned gs = (unsigned)((n + 255) / 256);
    emu::launch(k_group_count, dim3(std::min(gs, 3u)), dim3(256), st, tp, pr, jn, n, shift, row.data(), slot.data(),
                count.data(), work.data());
    unsigned long long all = 0, big = 0;
    int most = 0;
    for (long long g = 0; g < groups; g++) {
        start[g + 1] = start[g] + count[g];
        most = std::max(most, count[g]);
        for (int k = 0; k < count[g]; k++) {
            all += (unsigned long long)k;
            if (k >= half) big += (unsigned long long)k;
        }
    }
    if (start[groups] != n || work[0] != all || work[2] != big || (all && work[1] + 1 != (unsigned long long)most)) return 1;
    emu::launch(k_group_scatter, dim3(gs), dim3(256), tp, pr, jn, n, shift, least, row.data(), slot.data(), start.data(),
                pos[0].data(), key[0].data(), seg[0].data());
    if (!rank_all)
        emu::launch(k_group_tile, dim3((unsigned)((n + half - 1) / half)), dim3(1024), tp, pr, jn, n, shift, row.data(),
                    pos[0].data(), seg[0].data(), perm.data());
    if (!rank_all && most >= least)
        emu::launch(k_group_list, dim3(gs), dim3(256), seg[0].data(), n, least, list.data(), &work[3]);
    int bits = 1;
    while ((1ll << bits) <= maxcnt) bits++;
    const int words = group_passes(stride, shift, bits);
    if (rank_all || most >= least)
        for (int w = 0, cur = 0; w < words; w++, cur ^= 1)
            emu::launch(k_group_rank, dim3(40), dim3(256), tp, pr, jn, n, rank_all ? (const int *)nullptr : list.data(),
                        &work[3], pos[cur].data(), key[cur].data(), seg[cur].data(),
                        w + 1 < words ? pos[cur ^ 1].data() : perm.data(), key[cur ^ 1].data(), seg[cur ^ 1].data());

    // report order: molecule, templates in reverse, list position of level 0, kd
    // positions of the further levels
    std::vector<std::vector<int>> want(n);
    for (long long i = 0; i < n; i++) {
        const int p = pair[i];
        want[i] = {p / T, T - 1 - p % T, kidx[ent[i * stride]]};
        for (int l = 1; l < size[p % T]; l++)
            want[i].push_back(ent[i * stride + l] - lvl[(size_t)p * JAM_MAX_LEVELS + l].off);
    }
    std::vector<int> sorted(n);
    std::iota(sorted.begin(), sorted.end(), 0);
    std::sort(sorted.begin(), sorted.end(), [&](int a, int b) { return want[a] < want[b]; });
    std::map<std::pair<unsigned int, unsigned long long>, int> first;
    for (long long i = 0; i < n; i++) {
        int l = 1;
        first[{row[i] >> shift, group_key(tp, pr, jn, (int)i, row[i] & ((1u << shift) - 1u), shift, l)}]++;
    }
    long long shared = 0;
    for (auto &x : first)
        if (x.second > 1) shared += x.second;
    std::printf("%lld %d %d %lld\n", n, most, words, shared);
    return std::equal(sorted.begin(), sorted.end(), perm.begin()) ? 0 : 1;
}
