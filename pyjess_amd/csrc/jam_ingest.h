// jam_ingest.h -- PDB text to device molecules, on gfx950.
//
// The reference reads a PDB file line by line in Python (PDBMoleculeParser,
// src/pyjess/_io.py:68-103): ATOM records, and HETATM records unless skipped,
// become atoms (Atom.loads: fixed columns), up to the first ENDMDL record
// unless it is ignored; mmCIF data tags are an error. Molecule.__init__ then
// builds the residue-name index (ResIndex_create,
// patches/ResIndex.c.patch:34-119): atoms sorted by case-insensitive residue
// name, then serial number, grouped into one bucket per name.
//
// Here the texts of a batch of molecules (concatenated, each ending with a
// line feed) go through:
//   k_ing_count / k_ing_starts  line starts (after '\n', '\r\n' or a lone '\r',
//                               as Python's universal newlines read them),
//                               counted per block, scanned, written in order
//   k_ing_classify              record type of every line, text of every line,
//                               first ENDMDL and first mmCIF tag of every text
//   k_ing_select                atom records in order (a scan of 0/1 flags)
//   k_ing_parse                 thread per atom record: the fixed columns
//   k_residue_index             the residue-name index: workgroup per molecule,
//                               a stable counting sort by name (of atoms
//                               ordered by serial number before, where those
//                               descend: k_run_order, or radix passes)
// Numbers are parsed exactly: a decimal field of at most 19 significant
// digits and a power of ten up to 22 is one correctly rounded division or
// multiplication of two exact doubles (Clinger's fast path), which is what
// Python's float() returns; other numeric forms are reported as errors.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "jam_common.h"
#include "jam_wave.h"

namespace jam {

#define ING_BPT 16          // bytes per thread when splitting lines
#define ING_THREADS 256
#define ING_MAX_NAMES 2048  // distinct residue names per molecule

// line and record kinds
#define ING_OTHER 0
#define ING_ATOM 1
#define ING_HETATM 2
#define ING_ENDMDL 3
#define ING_MMCIF 4
#define ING_HEADER 5

// what the line split and the record kinds report beside them: whether any
// byte is above 0x7F, how many HEADER records there are, and of the first
// ING_HEADERS of them (in any order) line and offset
#define ING_HEADERS 256
#define ING_INFO_WORDS (2 + 2 * ING_HEADERS)

// most atoms at which serial numbers descend for k_run_order
#define ING_RUNS 64
#define RUN_CHAINS 4   // bisections side by side

// parse errors (bit flags of the per-atom error word)
#define ING_EBADFIELD 1     // a numeric field does not parse
#define ING_ENONASCII 2     // a byte above 0x7F in the first 80 columns

struct IngText {
    const unsigned char *buf;  // the texts, concatenated, each ending with '\n'
    long long n_bytes;
    const long long *text_off; // n_texts + 1
    int n_texts;
    int flags;                 // JAM_PDB_* of the ABI
};

__device__ static inline bool ing_line_start(const unsigned char *b, long long i)
{
    if (i == 0) return true;
    const unsigned char p = b[i - 1];
    return p == '\n' || (p == '\r' && b[i] != '\n');
}

// in-block exclusive scan of one value per thread (ING_THREADS threads)
__device__ static inline long long ing_block_scan(long long v, long long *lds, long long &total)
{
    const int t = threadIdx.x, lane = lane_id(), w = t / JAM_WAVE;
    long long x = v;
    for (int sh = 1; sh < JAM_WAVE; sh <<= 1) {
        const long long y = __shfl_up(x, sh, JAM_WAVE);
        if (lane >= sh) x += y;
    }
    if (lane == JAM_WAVE - 1) lds[w] = x;
    __syncthreads();
    long long base = 0;
    total = 0;
    for (int k = 0; k < ING_THREADS / JAM_WAVE; k++) {
        if (k < w) base += lds[k];
        total += lds[k];
    }
    __syncthreads();
    return base + x - v;
}

// Line starts of each block's ING_THREADS * ING_BPT bytes.
__global__ void __launch_bounds__(ING_THREADS) k_ing_count(IngText tx, long long *block_lines,
                                                          unsigned long long *info)
{
    __shared__ long long lds[ING_THREADS / JAM_WAVE];
    const long long b0 = ((long long)blockIdx.x * ING_THREADS + threadIdx.x) * ING_BPT;
    long long c = 0;
    bool high = false;
    for (int k = 0; k < ING_BPT; k++) {
        const long long i = b0 + k;
        if (i >= tx.n_bytes) break;
        if (ing_line_start(tx.buf, i)) c++;
        high |= tx.buf[i] > 0x7F;
    }
    if (ballot(high) != 0ull && lane_id() == 0) atomicOr(&info[0], 1ull);
    long long total;
    ing_block_scan(c, lds, total);
    if (threadIdx.x == 0) block_lines[blockIdx.x] = total;
}

// Writes the line starts in order (block_off: exclusive scan of block_lines).
__global__ void __launch_bounds__(ING_THREADS) k_ing_starts(IngText tx, const long long *block_off, long long *starts)
{
    __shared__ long long lds[ING_THREADS / JAM_WAVE];
    const long long b0 = ((long long)blockIdx.x * ING_THREADS + threadIdx.x) * ING_BPT;
    long long c = 0;
    for (int k = 0; k < ING_BPT; k++) {
        const long long i = b0 + k;
        if (i < tx.n_bytes && ing_line_start(tx.buf, i)) c++;
    }
    long long total;
    long long o = block_off[blockIdx.x] + ing_block_scan(c, lds, total);
    for (int k = 0; k < ING_BPT; k++) {
        const long long i = b0 + k;
        if (i < tx.n_bytes && ing_line_start(tx.buf, i)) starts[o++] = i;
    }
}

// end of line li (one past its last character, terminators excluded)
__device__ static inline long long ing_line_end(const IngText &tx, const long long *starts, long long n_lines,
                                                long long li)
{
    long long e = li + 1 < n_lines ? starts[li + 1] : tx.n_bytes;
    const long long s = starts[li];
    while (e > s && (tx.buf[e - 1] == '\n' || tx.buf[e - 1] == '\r')) e--;
    return e;
}

__device__ static inline int ing_text_of(const IngText &tx, long long pos)
{
    int lo = 0, hi = tx.n_texts;   // the last text whose start is <= pos
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (tx.text_off[mid] <= pos) lo = mid;
        else hi = mid;
    }
    return lo;
}

__device__ static inline unsigned char ing_lower(unsigned char c) { return (c >= 'A' && c <= 'Z') ? c + 32 : c; }

// Kind and text of every line; first ENDMDL and first mmCIF tag per text
// (first_endmdl, first_mmcif: n_texts words each, preset to n_lines).
__global__ void __launch_bounds__(ING_THREADS) k_ing_classify(IngText tx, const long long *starts, long long n_lines,
                                                             unsigned char *kind, int *text_of,
                                                             unsigned long long *first_endmdl,
                                                             unsigned long long *first_mmcif,
                                                             unsigned long long *info)
{
    const long long li = (long long)blockIdx.x * ING_THREADS + threadIdx.x;
    if (li >= n_lines) return;
    const long long s = starts[li], e = ing_line_end(tx, starts, n_lines, li);
    const unsigned char *p = tx.buf + s;
    const long long len = e - s;
    auto at = [&](int k) { return k < len ? p[k] : (unsigned char)0; };
    unsigned char k = ING_OTHER;
    if (at(0) == 'A' && at(1) == 'T' && at(2) == 'O' && at(3) == 'M') k = ING_ATOM;
    else if (at(0) == 'H' && at(1) == 'E' && at(2) == 'T' && at(3) == 'A' && at(4) == 'T' && at(5) == 'M') k = ING_HETATM;
    else if (at(0) == 'E' && at(1) == 'N' && at(2) == 'D' && at(3) == 'M' && at(4) == 'D' && at(5) == 'L') k = ING_ENDMDL;
    else if (at(0) == 'H' && at(1) == 'E' && at(2) == 'A' && at(3) == 'D' && at(4) == 'E' && at(5) == 'R') k = ING_HEADER;
    else if (len >= 5) {
        const unsigned char a = ing_lower(p[0]), b = ing_lower(p[1]), c = ing_lower(p[2]), d = ing_lower(p[3]);
        if (p[4] == '_' && ((a == 'd' && b == 'a' && c == 't' && d == 'a') || (a == 'l' && b == 'o' && c == 'o' && d == 'p')))
            k = ING_MMCIF;
    }
    kind[li] = k;
    const int t = ing_text_of(tx, s);
    text_of[li] = t;
    if (k == ING_ENDMDL) atomicMin(&first_endmdl[t], (unsigned long long)li);
    if (k == ING_MMCIF) atomicMin(&first_mmcif[t], (unsigned long long)li);
    if (k == ING_HEADER) {
        const unsigned long long h = atomicAdd(&info[1], 1ull);
        if (h < ING_HEADERS) {
            info[2 + 2 * h] = (unsigned long long)li;
            info[3 + 2 * h] = (unsigned long long)s;
        }
    }
}

// whether line li is an atom record the reference would read
__device__ static inline int ing_is_atom(const IngText &tx, const unsigned char *kind, const int *text_of,
                                         const unsigned long long *first_endmdl, long long li)
{
    const unsigned char k = kind[li];
    if (k != ING_ATOM && !(k == ING_HETATM && !(tx.flags & 1))) return 0;
    // records after the first ENDMDL are not read unless it is ignored
    if (!(tx.flags & 2) && (unsigned long long)li > first_endmdl[text_of[li]]) return 0;
    return 1;
}

// atom records per block of ING_THREADS lines
__global__ void __launch_bounds__(ING_THREADS) k_ing_select_count(IngText tx, const unsigned char *kind,
                                                                 const int *text_of,
                                                                 const unsigned long long *first_endmdl,
                                                                 long long n_lines, long long *block_atoms)
{
    __shared__ long long lds[ING_THREADS / JAM_WAVE];
    const long long li = (long long)blockIdx.x * ING_THREADS + threadIdx.x;
    const long long v = li < n_lines ? ing_is_atom(tx, kind, text_of, first_endmdl, li) : 0;
    long long total;
    ing_block_scan(v, lds, total);
    if (threadIdx.x == 0) block_atoms[blockIdx.x] = total;
}

// atom_line[a]: the line of atom record a, in order; line_atom[li]: the atom
// index of line li's record, or of the next record (the count before it)
__global__ void __launch_bounds__(ING_THREADS) k_ing_select(IngText tx, const unsigned char *kind, const int *text_of,
                                                           const unsigned long long *first_endmdl, long long n_lines,
                                                           const long long *block_off, long long *atom_line,
                                                           long long *line_atom)
{
    __shared__ long long lds[ING_THREADS / JAM_WAVE];
    const long long li = (long long)blockIdx.x * ING_THREADS + threadIdx.x;
    const int v = li < n_lines ? ing_is_atom(tx, kind, text_of, first_endmdl, li) : 0;
    long long total;
    const long long a = block_off[blockIdx.x] + ing_block_scan(v, lds, total);
    if (li < n_lines) line_atom[li] = a;
    if (v) atom_line[a] = li;
}

// per text: its first line and its first atom (n_texts + 1 entries each)
__global__ void k_ing_text_ranges(IngText tx, const long long *starts, long long n_lines, const long long *line_atom,
                                  const long long *n_atoms, long long *text_line, long long *text_atom)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t > tx.n_texts) return;
    long long lo = 0, hi = n_lines;   // first line starting at or after the text's first byte
    const long long pos = tx.text_off[t];
    while (lo < hi) {
        const long long mid = (lo + hi) >> 1;
        if (starts[mid] < pos) lo = mid + 1;
        else hi = mid;
    }
    text_line[t] = lo;
    text_atom[t] = lo < n_lines ? line_atom[lo] : (n_lines > 0 ? *n_atoms : 0);
}

// ---------------------------------------------------------------------------
// fixed columns of one record
// ---------------------------------------------------------------------------

__constant__ double ING_POW10[23] = {1e0,  1e1,  1e2,  1e3,  1e4,  1e5,  1e6,  1e7,  1e8,  1e9,  1e10, 1e11,
                                     1e12, 1e13, 1e14, 1e15, 1e16, 1e17, 1e18, 1e19, 1e20, 1e21, 1e22};

// str.strip()'s whitespace among ASCII bytes
__device__ static inline bool ing_space(unsigned char c) { return c == ' ' || (c >= 9 && c <= 13) || (c >= 28 && c <= 31); }

// int(field): optional sign, at least one digit, whitespace around
__device__ static inline bool ing_int(const unsigned char *f, int n, int &out)
{
    int i = 0;
    while (i < n && ing_space(f[i])) i++;
    bool neg = false;
    if (i < n && (f[i] == '+' || f[i] == '-')) neg = f[i++] == '-';
    long long v = 0;
    int digits = 0;
    while (i < n && f[i] >= '0' && f[i] <= '9') {
        v = v * 10 + (f[i++] - '0');
        if (++digits > 9) return false;   // fields are at most 5 characters
    }
    while (i < n && ing_space(f[i])) i++;
    if (digits == 0 || i != n) return false;
    out = (int)(neg ? -v : v);
    return true;
}

// float(field) for decimal forms: sign, digits with at most one point,
// optional exponent, whitespace around; exact (correctly rounded) when the
// significant digits fit 19 and the power of ten 22, else false
__device__ static inline bool ing_f64(const unsigned char *f, int n, double &out)
{
    int i = 0;
    while (i < n && ing_space(f[i])) i++;
    bool neg = false;
    if (i < n && (f[i] == '+' || f[i] == '-')) neg = f[i++] == '-';
    unsigned long long N = 0;
    int sig = 0, digits = 0, scale = 0;
    bool point = false;
    for (; i < n; i++) {
        const unsigned char c = f[i];
        if (c >= '0' && c <= '9') {
            digits++;
            if (N == 0 && c == '0') {
                if (point) scale--;
                continue;                      // leading zeros are not significant
            }
            if (++sig > 19) return false;
            N = N * 10 + (c - '0');
            if (point) scale--;
        } else if (c == '.' && !point) {
            point = true;
        } else {
            break;
        }
    }
    if (digits == 0) return false;
    if (i < n && (f[i] == 'e' || f[i] == 'E')) {
        i++;
        bool eneg = false;
        if (i < n && (f[i] == '+' || f[i] == '-')) eneg = f[i++] == '-';
        int ev = 0, ed = 0;
        while (i < n && f[i] >= '0' && f[i] <= '9') {
            ev = ev * 10 + (f[i++] - '0');
            if (++ed > 4) return false;
        }
        if (ed == 0) return false;
        scale += eneg ? -ev : ev;
    }
    while (i < n && ing_space(f[i])) i++;
    if (i != n) return false;
    double v;
    if (N == 0) {
        v = 0.0;
    } else {
        if (N >= (1ull << 53) || scale > 22 || scale < -22) return false;
        v = scale >= 0 ? (double)N * ING_POW10[scale] : (double)N / ING_POW10[-scale];
    }
    out = neg ? -v : v;
    return true;
}

// the per-atom arrays a parse fills
struct IngAtoms {
    double *xyz;             // 3 per atom
    uint32_t *name;          // 4 bytes, blanks and NUL as '_'
    uint32_t *resname;       // 3 bytes + NUL, blanks and NUL as '_'
    int *chain;              // chainID2 as a signed char value (what the search reads)
    unsigned char *chains;   // 2 per atom: chainID1, chainID2
    int *resseq, *serial;
    unsigned char *altloc, *icode;
    float *occupancy, *tempfactor;
    uint32_t *segid;         // 4 bytes, blanks and NUL as '_'
    unsigned short *element; // 2 bytes, blanks and NUL as '_'
    int *charge;
    unsigned int *err;       // per atom: ING_E* bits
    unsigned long long *first_err;   // device word: the first atom with an error (preset to n_atoms)
};

__device__ static inline unsigned char ing_tok(unsigned char c) { return (c == ' ' || c == 0) ? '_' : c; }

// Thread per atom record: Atom.loads (the PDB fixed columns, the line padded
// with blanks to 80 characters).
__global__ void __launch_bounds__(ING_THREADS) k_ing_parse(IngText tx, const long long *starts, long long n_lines,
                                                          const long long *atom_line, long long n_atoms, IngAtoms at)
{
    const long long a = (long long)blockIdx.x * ING_THREADS + threadIdx.x;
    if (a >= n_atoms) return;
    const long long li = atom_line[a];
    const long long s = starts[li], e = ing_line_end(tx, starts, n_lines, li);
    unsigned char col[80];
    unsigned int err = 0;
    const long long len = e - s;
#pragma unroll 8
    for (int k = 0; k < 80; k++) {
        const unsigned char c = k < len ? tx.buf[s + k] : (unsigned char)' ';
        if (c > 0x7F) err |= ING_ENONASCII;
        col[k] = c;
    }
    int serial = 0, resseq = 0;
    double x = 0.0, y = 0.0, z = 0.0, occ = 0.0, tf = 0.0;
    if (!ing_int(col + 6, 5, serial) || !ing_int(col + 22, 4, resseq) || !ing_f64(col + 30, 8, x) ||
        !ing_f64(col + 38, 8, y) || !ing_f64(col + 46, 8, z))
        err |= ING_EBADFIELD;
    // occupancy and temperature factor: blank is 0.0
    auto num = [&](int c0, int w, double &v) {
        int i = c0, j = c0 + w;
        while (i < j && ing_space(col[i])) i++;
        while (j > i && ing_space(col[j - 1])) j--;
        if (i == j) {
            v = 0.0;
            return true;
        }
        return ing_f64(col + i, j - i, v);
    };
    if (!num(54, 6, occ) || !num(60, 6, tf)) err |= ING_EBADFIELD;
    // charge: the stripped two columns read backwards ("2+" is +2), 0 when
    // that is not an integer
    int charge = 0;
    {
        int i = 78, j = 80;
        while (i < j && ing_space(col[i])) i++;
        while (j > i && ing_space(col[j - 1])) j--;
        unsigned char rev[2];
        const int m = j - i;
        for (int k = 0; k < m; k++) rev[k] = col[j - 1 - k];
        int v = 0;
        if (m > 0 && ing_int(rev, m, v)) charge = v;
    }
    at.xyz[3 * a + 0] = x;
    at.xyz[3 * a + 1] = y;
    at.xyz[3 * a + 2] = z;
    at.name[a] = ing_tok(col[12]) | (ing_tok(col[13]) << 8) | (ing_tok(col[14]) << 16) | ((uint32_t)ing_tok(col[15]) << 24);
    at.resname[a] = ing_tok(col[17]) | (ing_tok(col[18]) << 8) | (ing_tok(col[19]) << 16);
    at.chain[a] = (int)(signed char)col[21];
    at.chains[2 * a + 0] = col[20];
    at.chains[2 * a + 1] = col[21];
    at.resseq[a] = resseq;
    at.serial[a] = serial;
    at.altloc[a] = col[16];
    at.icode[a] = col[26];
    at.occupancy[a] = (float)occ;
    at.tempfactor[a] = (float)tf;
    at.segid[a] = ing_tok(col[72]) | (ing_tok(col[73]) << 8) | (ing_tok(col[74]) << 16) | ((uint32_t)ing_tok(col[75]) << 24);
    at.element[a] = (unsigned short)(ing_tok(col[76]) | (ing_tok(col[77]) << 8));
    at.charge[a] = charge;
    at.err[a] = err;
    if (err) atomicMin(at.first_err, (unsigned long long)a);
}

// ---------------------------------------------------------------------------
// residue-name index
// ---------------------------------------------------------------------------

// Atoms whose serial number is below that of the atom before them in their
// text: their number to *n_down, the first ING_RUNS of them (in any order) to
// down.
__global__ void __launch_bounds__(ING_THREADS) k_ing_descends(long long n_atoms, const int *serial,
                                                             const long long *atom_line, const int *text_of,
                                                             unsigned long long *n_down, int *down)
{
    const long long a = (long long)blockIdx.x * ING_THREADS + threadIdx.x;
    const bool d = a > 0 && a < n_atoms && serial[a] < serial[a - 1] && text_of[atom_line[a]] == text_of[atom_line[a - 1]];
    const unsigned long long m = ballot(d);
    if (m == 0ull) return;
    unsigned long long k = 0;
    if (lane_id() == 0) k = atomicAdd(n_down, (unsigned long long)__popcll(m));
    k = __shfl(k, 0, JAM_WAVE) + rank_below(m);
    if (d && k < ING_RUNS) down[k] = (int)a;
}

// the molecule that atom a of the batch belongs to: the last that starts at or before it
__device__ static inline int molecule_of(const int *atom_off, int n_mols, long long a)
{
    int lo = 0, hi = n_mols;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (atom_off[mid] <= a) lo = mid;
        else hi = mid;
    }
    return lo;
}

// Molecule-local indices of every molecule's atoms by serial number, ties in
// input order, at its positions in order, where the serial numbers descend at the few
// atoms `down` (in any order): an atom's place is the number of atoms before it in
// each ascending run, by bisection (RUN_CHAINS runs at once). Bound by the chains
// of a bisection (17 loads for 100,000 atoms), which the other waves hide. With
// k_visited_names: a text of 100,000 atoms that wraps once 1.08 (radix passes) -> 0.89
// ms, of 2 M atoms in 21 runs 12.2 -> 11.0 ms; upload of 400,000 atoms in 5 runs
// 12.6 (sorted on the host) -> 2.1 ms.
__global__ void __launch_bounds__(ING_THREADS) k_run_order(const int *atom_off, int n_mols, const int *serial,
                                                          const int *down, int n_down, int *order)
{
    __shared__ int first[ING_RUNS];
    const int t = threadIdx.x;
    if (t < n_down) {
        const int v = down[t];
        int k = 0;
        for (int q = 0; q < n_down; q++) k += down[q] < v;
        first[k] = v;
    }
    __syncthreads();
    const long long a = (long long)blockIdx.x * ING_THREADS + t;
    if (a >= atom_off[n_mols]) return;
    const int m = molecule_of(atom_off, n_mols, a);
    const int a0 = atom_off[m], a1 = atom_off[m + 1], s = serial[a];
    // run r of the molecule: [first[k0 + r - 1], first[k0 + r]), a0 and a1 at its ends
    int k0 = 0, k1;
    while (k0 < n_down && first[k0] <= a0) k0++;
    for (k1 = k0; k1 < n_down && first[k1] < a1;) k1++;
    unsigned at = (unsigned)a0;   // (sums of places, which pass the range of an int)
    for (int r0 = k0; r0 <= k1; r0 += RUN_CHAINS) {
        int x[RUN_CHAINS], y[RUN_CHAINS];
        bool upto[RUN_CHAINS];   // an earlier run counts up to s, a later one below s
#pragma unroll
        for (int u = 0; u < RUN_CHAINS; u++) {
            const int r = r0 + u;
            const int begin = r == k0 ? a0 : r <= k1 ? first[r - 1] : a1, end = r < k1 ? first[r] : a1;
            upto[u] = begin <= a;
            x[u] = begin;
            y[u] = end;
            at -= (unsigned)begin;
            if (a >= begin && a < end) x[u] = y[u] = (int)a;
        }
        for (bool more = true; more;) {
            more = false;
#pragma unroll
            for (int u = 0; u < RUN_CHAINS; u++) {
                if (x[u] >= y[u]) continue;
                const int mid = x[u] + ((y[u] - x[u]) >> 1), v = serial[mid];
                if (upto[u] ? v <= s : v < s) x[u] = mid + 1;
                else y[u] = mid;
                more = true;
            }
        }
#pragma unroll
        for (int u = 0; u < RUN_CHAINS; u++) at += (unsigned)x[u];
    }
    order[at] = (int)a - a0;
}

// Sort key of every atom: its molecule, then its serial number, which a stable
// sort orders as k_residue_index visits atoms whose serial numbers descend
// at many places; the value is the atom's index.
__global__ void __launch_bounds__(ING_THREADS) k_serial_keys(const int *atom_off, int n_mols, const int *serial,
                                                            unsigned long long *key, int *val)
{
    const long long a = (long long)blockIdx.x * ING_THREADS + threadIdx.x;
    if (a >= atom_off[n_mols]) return;
    key[a] = ((unsigned long long)(unsigned int)molecule_of(atom_off, n_mols, a) << 32) |
             ((unsigned int)serial[a] ^ 0x80000000u);
    val[a] = (int)a;
}

// order[i]: the molecule-local index of the i-th sorted atom (a molecule's atoms
// keep its positions)
__global__ void __launch_bounds__(ING_THREADS) k_sorted_order(const int *atom_off, int n_mols, const int *sorted,
                                                             int *order)
{
    const long long i = (long long)blockIdx.x * ING_THREADS + threadIdx.x;
    if (i >= atom_off[n_mols]) return;
    order[i] = sorted[i] - atom_off[molecule_of(atom_off, n_mols, i)];
}

// out[k] = (int)in[k]
__global__ void k_ing_narrow(const long long *in, int n, int *out)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) out[k] = (int)in[k];
}

// The residue names of every molecule's atoms in the order in which
// k_residue_index visits them: gathered by the whole device, as one molecule's
// workgroup alone takes 1.4 ms more for 2 M atoms of 21 interleaved runs.
__global__ void __launch_bounds__(ING_THREADS) k_visited_names(const int *atom_off, int n_mols, const uint32_t *resname,
                                                              const int *order, uint32_t *visited)
{
    const long long i = (long long)blockIdx.x * ING_THREADS + threadIdx.x;
    if (i >= atom_off[n_mols]) return;
    visited[i] = resname[atom_off[molecule_of(atom_off, n_mols, i)] + order[i]];
}

// The residue-name index of a batch in one launch (ResIndex_create,
// patches/ResIndex.c.patch:34-119): a workgroup per molecule. The molecule's
// distinct upper-cased names go through an LDS hash set and a bitonic sort
// (groups ordered by key value, which the candidate kernels' binary search
// expects); then each of the 16 waves takes a contiguous 16th of the atoms,
// counts its atoms per name, and after a scan over (name, wave) walks them
// again, 64 at a time, to their places: a lane's rank among the lanes of its
// name comes from one ballot per bit of the name's number, so the counting
// sort is stable and its second walk needs no workgroup barrier.
// `order`, where given, is the order in which a molecule's atoms are visited
// (its molecule-local indices by serial number, ties in input order), and
// `visited` their names in that order (else resname); without
// it they are visited as they come, which is the same thing for serial numbers
// that never descend. Either way atoms end up by (name, serial, input order).
//
// keys / starts: the k-th name of molecule m and the first position of its
// group at [atom_off[m] + k] (a molecule has no more names than atoms).
// n_names[m] = -1 where a molecule has more than MAXN names, or one whose four
// bytes are all 0xFF (the empty slot's mark).
//
// Bound by latency (two walks with one dependent load each and ~10 LDS steps
// per 64 atoms of a wave) and by the waves in flight: 2 workgroups of 16 waves
// per CU at MAXN = 256 (19 KB of LDS; 152 KB at ING_MAX_NAMES, for molecules
// of more names). One launch for all molecules instead of
// a host sort: jam_molecules_create of 256 molecules (1.2 M atoms) 39.6 -> 3.2
// ms, of 100,000 atoms 2.2 -> 0.57 ms, of 2,000 atoms 0.22 -> 0.07 ms, with
// the upload through pinned memory that came with it. A single large molecule has
// one workgroup all the same: of 2 M atoms 57 -> 8.9 ms, parsed from text 11.0 ms
// with this index and with the grid-wide sort before it.
#define IDX_THREADS 1024
#define IDX_WAVES (IDX_THREADS / JAM_WAVE)
#define IDX_MAX_NAMES 256

template <int MAXN>
__global__ void __launch_bounds__(IDX_THREADS) k_residue_index(const int *atom_off, const uint32_t *resname,
                                                               const uint32_t *visited, const int *order, int *perm, uint32_t *keys,
                                                               int *starts, int *n_names)
{
    constexpr int SLOTS = 2 * MAXN;   // open addressing at half load at most
    constexpr uint32_t EMPTY = 0xFFFFFFFFu;
    __shared__ uint32_t slot[SLOTS];
    __shared__ uint32_t list[MAXN];
    __shared__ int run[IDX_WAVES][MAXN];   // per wave and name: atoms, then the next position
    __shared__ int count, refused;
    const int m = blockIdx.x, t = threadIdx.x, lane = lane_id(), w = t / JAM_WAVE;
    for (int k = t; k < SLOTS; k += IDX_THREADS) slot[k] = EMPTY;
    if (t == 0) {
        count = 0;
        refused = 0;
    }
    __syncthreads();
    const int a0 = atom_off[m], n_atoms = atom_off[m + 1] - a0;
    // distinct names: the first atom of a run of equal names (as stored)
    // enters it for the run
    for (int i = t; i < n_atoms; i += IDX_THREADS) {
        const uint32_t key = jam_upper4(resname[a0 + i]);
        if (i > 0 && jam_upper4(resname[a0 + i - 1]) == key) continue;
        if (key == EMPTY) {
            refused = 1;
            continue;
        }
        uint32_t h = (key * 2654435761u) >> 7;
        for (int probe = 0; probe < SLOTS; probe++) {
            h &= SLOTS - 1;
            const uint32_t old = atomicCAS(&slot[h], EMPTY, key);
            if (old == EMPTY) {
                const int c = atomicAdd(&count, 1);
                if (c < MAXN) list[c] = key;
                break;
            }
            if (old == key) break;
            h++;
        }
        if (count > MAXN) break;
    }
    __syncthreads();
    const int n = count;
    if (n > MAXN || refused) {
        if (t == 0) n_names[m] = -1;
        return;
    }
    int n2 = 1, bits = 0;
    while (n2 < n) {
        n2 <<= 1;
        bits++;
    }
    for (int k = n + t; k < n2; k += IDX_THREADS) list[k] = EMPTY;
    for (int k = t; k < IDX_WAVES * n; k += IDX_THREADS) run[k / n][k % n] = 0;
    __syncthreads();
    for (int k = 2; k <= n2; k <<= 1) {
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int i = t; i < n2; i += IDX_THREADS) {
                const int ixj = i ^ j;
                if (ixj > i) {
                    const uint32_t u = list[i], v = list[ixj];
                    if ((u > v) == ((i & k) == 0)) {
                        list[i] = v;
                        list[ixj] = u;
                    }
                }
            }
            __syncthreads();
        }
    }
    // this wave's part of the atoms, a multiple of 64
    const int per = ((n_atoms + IDX_THREADS - 1) / IDX_THREADS) * JAM_WAVE;
    const int begin = min(w * per, n_atoms), end = min(begin + per, n_atoms);
    // the i-th visited atom (molecule-local) and the number of its name
    auto visit = [&](int i, int &atom, int &b) {
        atom = order ? order[a0 + i] : i;
        const uint32_t key = jam_upper4(visited[a0 + i]);
        int lo = 0, hi = n - 1;   // the last name <= key is key itself
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (list[mid] <= key) lo = mid;
            else hi = mid - 1;
        }
        b = lo;
    };
    for (int i = begin + lane; i < end; i += JAM_WAVE) {
        int atom, b;
        visit(i, atom, b);
        atomicAdd(&run[w][b], 1);
    }
    __syncthreads();
    // where each name's group starts, and in it each wave's part
    if (t < JAM_WAVE) {
        int carry = 0;
        for (int b0 = 0; b0 < n; b0 += JAM_WAVE) {
            const int b = b0 + lane;
            int v = 0;
            if (b < n)
                for (int q = 0; q < IDX_WAVES; q++) v += run[q][b];
            int x = v;
            for (int sh = 1; sh < JAM_WAVE; sh <<= 1) {
                const int y = __shfl_up(x, sh, JAM_WAVE);
                if (lane >= sh) x += y;
            }
            if (b < n) {
                int at = carry + x - v;
                keys[a0 + b] = list[b];
                starts[a0 + b] = at;
                for (int q = 0; q < IDX_WAVES; q++) {
                    const int c = run[q][b];
                    run[q][b] = at;
                    at += c;
                }
            }
            carry += __shfl(x, JAM_WAVE - 1, JAM_WAVE);
        }
        if (lane == 0) n_names[m] = n;
    }
    __syncthreads();
    for (int i0 = begin; i0 < end; i0 += JAM_WAVE) {
        const int i = i0 + lane;
        const bool ok = i < end;
        int atom = 0, b = 0;
        if (ok) visit(i, atom, b);
        unsigned long long peers = ballot(ok);
        for (int q = 0; q < bits; q++) {
            const bool bit = ((b >> q) & 1) != 0;
            const unsigned long long x = ballot(bit);
            peers &= bit ? x : ~x;
        }
        const int rank = rank_below(peers);
        int at = 0;
        if (ok) at = run[w][b];
        wave_sync();
        if (ok) {
            perm[a0 + at + rank] = atom;
            if (rank == 0) run[w][b] = at + __popcll(peers);
        }
        wave_sync();
    }
}

// The names and ranges of every molecule's groups, packed (res_off: the
// exclusive scan of n_names).
__global__ void __launch_bounds__(ING_THREADS) k_index_ranges(const int *atom_off, const uint32_t *keys,
                                                             const int *starts, const int *res_off, uint32_t *res_key,
                                                             int *res_begin, int *res_end)
{
    const int m = blockIdx.x, a0 = atom_off[m], n_atoms = atom_off[m + 1] - a0;
    const int r0 = res_off[m], n = res_off[m + 1] - r0;
    for (int k = threadIdx.x; k < n; k += ING_THREADS) {
        res_key[r0 + k] = keys[a0 + k];
        res_begin[r0 + k] = starts[a0 + k];
        res_end[r0 + k] = k + 1 < n ? starts[a0 + k + 1] : n_atoms;
    }
}

// A chain byte per atom to the (sign-extended) word that the search compares.
__global__ void __launch_bounds__(ING_THREADS) k_chain_words(const signed char *in, long long n, int *out)
{
    const long long i = (long long)blockIdx.x * ING_THREADS + threadIdx.x;
    if (i < n) out[i] = in[i];
}

}  // namespace jam
