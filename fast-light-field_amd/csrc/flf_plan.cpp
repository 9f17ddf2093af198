// Host-side planning for the light-field projector: Fourier shapes, radix
// plans and the orbit/item tables of the multiply-accumulate kernel.
//
// Items.  Every half-plane output bin k (k1 <= fX/2) of one plane needs the
// stored spectra at k, (-k0, k1) [row flip], (k1, k0) and (-k1, k0)
// [transposes; square grids only].  Grouping those bins into one item lets
// the kernel read each stored value once and use it for all of them:
//   square     quad  P0=(p0,p1) P1=(-p0,p1) P2=(p1,p0) P3=(-p1,p0),
//              base p in D = {0 <= p1 <= p0 <= f/2}
//   non-square pair  P0=(p0,p1) P1=(-p0,p1), p0 <= fY/2, p1 <= fX/2
// Every half-plane bin is the slot of exactly one item (slots of the same item
// may coincide on the boundaries of D; only the first writes its bin).
//
// Orbits.  The small FFTs S_{b,a} are periodic with the reduced grid r = f/N,
// so the kernel needs S only at the residues (k mod r) of its items' bins.
// Items are grouped by the orbit of their base residue under the symmetry
// group of the item (the dihedral group of the reduced square grid, or the
// sign flips of each axis for non-square grids): one orbit has at most 8
// residues and about N*N items, so a workgroup holds the N*N small-FFT values
// of <= 8 residues in LDS and streams the spectra of its items exactly once.
//
// Aliases.  A bin k = kt + m*r is written with kt the centred residue
// (|kt| < r/2) and m its alias; for the residue r/2 (r even) kt = 0 and m is
// a half integer.  Under this convention negating k negates m exactly, which
// is what lets all flip/transposition phases reduce to per-offset constants
// (folded into the s-table) and per-bin constants (the four classes).
#include "flf_plan.h"

#include <algorithm>
#include <array>

namespace flf {

static int max_prime_factor(int n) {
    int m = 1;
    for (int p = 2; p * p <= n; ++p)
        while (n % p == 0) { m = std::max(m, p); n /= p; }
    if (n > 1) m = std::max(m, n);
    return m;
}

int smooth5_at_least(int n) {
    int m = std::max(n, 1);
    while (m > 1 && max_prime_factor(m) > 5) ++m;
    return m;
}

int fourier_len(int s1, int s2, int N) {
    int need = s1 + s2 - 1;
    int red = (need + N - 1) / N;
    return N * smooth5_at_least(red);
}

// Plan of a 5-smooth length with radices up to 12: as few passes as possible,
// then the least sum of radices (work), largest first.
static bool shortest_plan(int L, RadixPlan& rp) {
    const int radices[9] = {2, 3, 4, 5, 6, 8, 9, 10, 12};
    std::vector<std::array<int, 3>> best(L + 1, {1 << 20, 0, 0});      // passes, sum, last radix
    best[1] = {0, 0, 0};
    for (int m = 2; m <= L; ++m) {
        if (L % m) continue;
        for (int R : radices)
            if (m % R == 0) {
                const std::array<int, 3> b{best[m / R][0] + 1, best[m / R][1] + R, R};
                if (b < best[m]) best[m] = b;
            }
    }
    if (best[L][0] > FLF_MAX_RADIX_PASSES - 1) return false;
    rp.L = L;
    rp.n = 0;
    for (int m = L; m > 1; m /= best[m][2]) rp.r[rp.n++] = best[m][2];
    std::sort(rp.r, rp.r + rp.n);
    std::reverse(rp.r, rp.r + rp.n);
    return true;
}

bool make_radix_plan(int L, RadixPlan& rp, bool wide, int order) {
    rp.L = L;
    rp.n = 0;
    int m = L;
    // Block-level transforms use radices 2..5, wave-level ones 8 and 6 too.
    // Orders 2 and 3 change the radices of wave-level plans only: the
    // block-level kernels size their butterfly registers from the plan's
    // radices (fft_batch_cap).
    const int narrow[4] = {4, 2, 3, 5};
    const int wider[4][6] = {{8, 6, 4, 5, 3, 2}, {8, 6, 4, 5, 3, 2}, {6, 4, 5, 3, 2, 0}, {5, 3, 8, 6, 4, 2}};
    if (order < 0 || order >= FLF_RADIX_ORDERS) return false;
    const int* list = wide ? wider[order] : narrow;
    const int nlist = wide ? 6 : 4;
    for (int k = 0; k < nlist; ++k) {
        const int R = list[k];
        if (R == 0) break;
        while (m % R == 0) {
            if (rp.n >= FLF_MAX_RADIX_PASSES) return false;
            rp.r[rp.n++] = R;
            m /= R;
        }
    }
    if (order == 1) std::reverse(rp.r, rp.r + rp.n);
    // One odd prime factor above 5 (a lenslet pitch such as 7, 13 or 19) is
    // taken as the last pass, the only position where a radix-P butterfly
    // writes onto its own inputs (see stockham_pass_prime, wave_pass_prime).
    if (m > 5 && m <= FLF_PRIME_RADIX_MAX && max_prime_factor(m) == m) {
        if (rp.n >= FLF_MAX_RADIX_PASSES) return false;
        rp.r[rp.n++] = m;
        m = 1;
    }
    return m == 1;
}

bool make_wave_plan(int L, RadixPlan& rp, int order) {
    // 3 or 4 passes (LDS round trips) instead of 4 or 5 at most lengths of 700
    // to 1800 (8 frames of 1455^2 x 41 planes: columns 2.85 -> 2.50 ms).
    if (order < 0 || order > 1) return make_radix_plan(L, rp, true, order);
    int m = L, smooth = 1;
    for (int R : {2, 3, 5})
        while (m % R == 0) { m /= R; smooth *= R; }
    if (!shortest_plan(smooth, rp)) return false;
    rp.L = L;
    if (order == 1) std::reverse(rp.r, rp.r + rp.n);
    if (m == 1) return true;
    if (m <= 5 || m > FLF_PRIME_RADIX_MAX || max_prime_factor(m) != m) return false;
    rp.r[rp.n++] = m;
    return true;
}

bool make_reduced_plan(int L, RadixPlan& rp, int order) {
    if (L > 128 || order < 0 || order >= FLF_RADIX_ORDERS || !shortest_plan(L, rp)) return false;
    if (order == 1) std::reverse(rp.r, rp.r + rp.n);
    return true;
}

// Half-unit alias of coordinate x on an axis of length N*r.
static int alias2(int x, int r, int N) {
    int k = x % r, m = x / r;
    if (2 * k < r) return (2 * m) % (2 * N);
    if (2 * k > r) return (2 * (m + 1)) % (2 * N);
    return (2 * m + 1) % (2 * N);
}

std::string build_grid_tables(int N, int fY, int fX, GridTables& gt) {
    if (N % 2 == 0 || N < 3 || N > FLF_MAX_N) return "Nnum must be odd and in [3, 31]";
    if (fY % N || fX % N) return "Fourier grid must be a multiple of Nnum";
    gt = GridTables();
    gt.fY = fY;
    gt.fX = fX;
    gt.rY = fY / N;
    gt.rX = fX / N;
    gt.rfX = fX / 2 + 1;
    gt.square = (fY == fX);
    gt.slots = gt.square ? 4 : 2;
    const int h = (N + 1) / 2, c = N / 2;

    // Stored spectra order (must match the category loops of k_mac).
    gt.u_bu.push_back(c); gt.u_au.push_back(c);
    if (gt.square) {
        for (int b = 0; b < c; ++b) { gt.u_bu.push_back(b); gt.u_au.push_back(b); }   // (b, b)
        for (int b = 0; b < c; ++b) { gt.u_bu.push_back(b); gt.u_au.push_back(c); }   // (b, c)
        for (int b = 0; b < c; ++b)
            for (int a = b + 1; a < c; ++a) { gt.u_bu.push_back(b); gt.u_au.push_back(a); }
    } else {
        for (int b = 0; b < c; ++b) { gt.u_bu.push_back(b); gt.u_au.push_back(c); }   // (b, c)
        for (int a = 0; a < c; ++a) { gt.u_bu.push_back(c); gt.u_au.push_back(a); }   // (c, a) = transpose of (a, c)
        for (int b = 0; b < c; ++b)
            for (int a = 0; a < c; ++a) { gt.u_bu.push_back(b); gt.u_au.push_back(a); }
    }
    gt.nu = (int)gt.u_bu.size();
    if (gt.nu != (gt.square ? h * (h + 1) / 2 : h * h)) return "internal: spectrum count";

    // Uses of each stored spectrum, in the order of the kernel's use types:
    // identity, both flips, row flip (N-1-b), column flip (N-1-a), then the
    // same four for the transposed PSF (py_light_field.cpp:1514-1560).
    const int NN = N * N;
    gt.nuse = gt.square ? 8 : 4;
    int present = 0;
    for (int u = 0; u < gt.nu; ++u) {
        const int bu = gt.u_bu[u], au = gt.u_au[u], bb = N - 1 - bu, ab = N - 1 - au;
        const bool mx = bu != c, my = au != c, tr = gt.square && au != bu;
        int o[8] = {bu * N + au,
                    (mx && my) ? bb * N + ab : NN,
                    mx ? bb * N + au : NN,
                    my ? bu * N + ab : NN,
                    tr ? au * N + bu : NN,
                    (tr && my && mx) ? ab * N + bb : NN,
                    (tr && my) ? ab * N + bu : NN,
                    (tr && mx) ? au * N + bb : NN};
        for (int q = 0; q < gt.nuse; ++q) {
            gt.uoff.push_back(o[q]);
            present += o[q] < NN;
        }
    }
    if (present != NN) return "internal: uses do not cover every offset once";
    // Pair types: the two uses that read the same slot of an item, one plain
    // and one conjugated (k_mac).
    const int plain[4] = {0, 2, 4, 7}, conj[4] = {1, 3, 5, 6};
    for (int u = 0; u < gt.nu; ++u)
        for (int pt = 0; pt < gt.slots; ++pt)
            for (int w = 0; w < 2; ++w) {
                const int off = gt.uoff[u * gt.nuse + (w == 0 ? plain[pt] : conj[pt])];
                gt.pairs.push_back(off < NN ? off * 8 + (off / N > c ? 1 : 0) + (off % N > c ? 2 : 0) : 4);
            }

    const int rY = gt.rY, rX = gt.rX, rfX = gt.rfX;
    // Residue, its negative and the half-unit alias of every coordinate.
    struct Axis { std::vector<int> res, neg; std::vector<unsigned char> al; };
    auto axis = [N](int f, int r) {
        Axis ax;
        for (int k = 0; k < f; ++k) {
            ax.res.push_back(k % r);
            ax.neg.push_back((r - k % r) % r);
            ax.al.push_back((unsigned char)alias2(k, r, N));
        }
        return ax;
    };
    const Axis aY = axis(fY, rY), aX = axis(fX, rX);
    // Orbit of a base: the least index among its residue's images (mirroring an
    // axis and, square grids, swapping the two).
    auto canon = [&](int p0, int p1) {
        const int a0 = std::min(aY.res[p0], aY.neg[p0]), a1 = std::min(aX.res[p1], aX.neg[p1]);
        return gt.square ? std::min(a0, a1) * rX + std::max(a0, a1) : a0 * rX + a1;
    };

    // Collect item bases per orbit (ordered by orbit key for determinism).
    std::vector<std::vector<std::pair<int, int>>> orbit_items((size_t)rY * rX);
    if (gt.square) {
        const int half = fY / 2;
        for (int p0 = 0; p0 <= half; ++p0)
            for (int p1 = 0; p1 <= p0; ++p1)
                orbit_items[canon(p0, p1)].push_back({p0, p1});
    } else {
        for (int p0 = 0; p0 <= fY / 2; ++p0)
            for (int p1 = 0; p1 <= fX / 2; ++p1)
                orbit_items[canon(p0, p1)].push_back({p0, p1});
    }

    gt.max_res = 0;
    for (size_t key = 0; key < orbit_items.size(); ++key) {
        auto& bases = orbit_items[key];
        if (bases.empty()) continue;
        // Residue list of the orbit in canonical order: the residues of the
        // first item's slots (its base residue k and the row-negated /
        // transposed ones), then their negatives.  The small-FFT kernel stores
        // S at the first half only; the MAC gets the second half by
        // conjugation (S(-k) = conj S(k) for real input).
        std::vector<std::pair<int, int>> res;
        std::array<int, 8> rkey;                                 // res as k0 * rX + k1
        {
            const int k0 = bases[0].first % rY, k1 = bases[0].second % rX;
            const int n0 = (rY - k0) % rY, n1 = (rX - k1) % rX;
            if (gt.square) {
                res = {{k0, k1}, {n0, k1}, {k1, k0}, {n1, k0}, {n0, n1}, {k0, n1}, {n1, n0}, {k1, n0}};
            } else {
                res = {{k0, k1}, {n0, k1}, {n0, n1}, {k0, n1}};
            }
            for (size_t q = 0; q < res.size(); ++q) rkey[q] = res[q].first * rX + res[q].second;
        }
        // An item may take the base of its transposed bin (square: slots 2, 3,
        // 0, 1) or of its negated row (non-square: slots 1, 0) just as well;
        // its class is then the partner of its own.
        auto make_item = [&](int p0, int p1, ItemDesc& it) -> const char* {
            int K0[4], K1[4];
            K0[0] = p0; K1[0] = p1;
            K0[1] = (fY - p0) % fY; K1[1] = p1;
            if (gt.square) {
                K0[2] = p1; K1[2] = p0;
                K0[3] = (fY - p1) % fY; K1[3] = p0;
            }
            it = ItemDesc{};
            it.writemask = 0;
            for (int j = 0; j < 4; ++j) {
                if (j >= gt.slots) {
                    it.pos[j] = it.pos[0]; it.res[j] = it.res[0]; it.m2[j] = it.m2[0]; it.n2[j] = it.n2[0];
                    continue;
                }
                if (K1[j] < 0 || K1[j] >= rfX) return "internal: slot outside half plane";
                it.pos[j] = K0[j] * rfX + K1[j];
                bool dup = false;
                for (int i = 0; i < j; ++i) dup |= (it.pos[i] == it.pos[j]);
                if (!dup) it.writemask |= (1 << j);
                const int rr = aY.res[K0[j]] * rX + aX.res[K1[j]], nr = (int)res.size();
                int ri = 0;
                while (ri < nr && rkey[ri] != rr) ++ri;
                if (ri == nr) return "internal: slot residue outside its orbit";
                it.res[j] = (unsigned char)ri;
                it.m2[j] = aY.al[K0[j]];
                it.n2[j] = aX.al[K1[j]];
            }
            return nullptr;
        };
        std::vector<ItemDesc> its;
        its.reserve(bases.size());
        // Classes (residue tuples, ascending) and their sizes: at most 8.
        typedef std::pair<unsigned, int> Class;
        auto class_of = [](const ItemDesc& it) {
            return (unsigned)it.res[0] << 24 | (unsigned)it.res[1] << 16 | (unsigned)it.res[2] << 8 | it.res[3];
        };
        std::vector<Class> size;
        auto find = [&size](unsigned c) {
            return std::find_if(size.begin(), size.end(), [c](const Class& x) { return x.first == c; });
        };
        for (auto& bp : bases) {
            ItemDesc it;
            if (const char* e = make_item(bp.first, bp.second, it)) return e;
            its.push_back(it);
            const unsigned c = class_of(it);
            auto f = find(c);
            if (f == size.end())
                size.push_back({c, 1});
            else
                ++f->second;
        }
        std::sort(size.begin(), size.end());
        // Tiles hold FLF_TILE items of one class: a class's items past its last
        // full tile move to the partner class if they fit into the open tile
        // there (at N = 15 one class of 36 and its partner of 28 become two of
        // 32: 8 tiles per orbit instead of 9, one workgroup instead of two).
        for (auto& kv : size) {
            const int rest = kv.second % FLF_TILE;
            if (kv.second <= FLF_TILE || rest == 0) continue;
            int left = rest;
            bool fits = false;
            for (size_t q = its.size(); q-- > 0 && left > 0;) {
                if (class_of(its[q]) != kv.first) continue;
                ItemDesc alt;
                const int p0 = bases[q].first, p1 = bases[q].second;
                if (const char* e = make_item(gt.square ? p1 : (fY - p0) % fY, gt.square ? p0 : p1, alt)) return e;
                const unsigned other = class_of(alt);
                if (other == kv.first) break;
                if (left == rest) {
                    auto f = find(other);
                    fits = f != size.end() && f->second % FLF_TILE != 0 && f->second % FLF_TILE + rest <= FLF_TILE;
                }
                if (!fits) break;
                its[q] = alt;
                ++find(other)->second;
                --kv.second;
                --left;
            }
        }
        gt.max_res = std::max(gt.max_res, (int)res.size());
        // Order by residue tuple (residue class): the MAC works on tiles of one
        // class, one per wave.
        std::vector<ItemDesc> sorted;
        sorted.reserve(its.size());
        for (const Class& c : size)
            for (const ItemDesc& it : its)
                if (class_of(it) == c.first) sorted.push_back(it);
        its.swap(sorted);
        // Tiles: runs of one residue class, at most FLF_TILE items each; at
        // most FLF_CHUNK_TILES of them (and FLF_CHUNK_MAX items) per chunk.
        size_t s = 0;
        while (s < its.size()) {
            ChunkDesc ch{};
            ch.item_base = (long long)gt.items.size();
            ch.n_res = (int)res.size();
            for (int q = 0; q < FLF_MAX_RES; ++q) {
                ch.res0[q] = q < ch.n_res ? res[q].first : 0;
                ch.res1[q] = q < ch.n_res ? res[q].second : 0;
            }
            ch.tile_base = (int)gt.tiles.size();
            while (s < its.size() && ch.n_tiles < FLF_CHUNK_TILES) {
                const ItemDesc& first = its[s];
                size_t e = s;
                while (e < its.size() && e - s < FLF_TILE && std::equal(its[e].res, its[e].res + 4, first.res)) ++e;
                if (ch.n_items + (int)(e - s) > FLF_CHUNK_MAX) break;
                TileDesc td{};
                td.start = ch.n_items;
                td.count = (int)(e - s);
                for (int j = 0; j < 4; ++j) td.res[j] = first.res[j];
                gt.tiles.push_back(td);
                gt.items.insert(gt.items.end(), its.begin() + s, its.begin() + e);
                ch.n_items += td.count;
                ch.n_tiles += 1;
                s = e;
            }
            gt.max_items = std::max(gt.max_items, ch.n_items);
            gt.chunks.push_back(ch);
        }
    }
    // The item slot that writes each half-plane bin, exactly one, then the bins'
    // places within their chunks: counted over the bins in (k1, k0) order.
    std::vector<int> owner((size_t)fY * rfX, -1), chunk_of(gt.items.size());
    std::vector<int> row(fY);
    for (size_t i = 0; i < gt.items.size(); ++i) {
        const ItemDesc& it = gt.items[i];
        for (int j = 0; j < gt.slots; ++j)
            if ((it.writemask >> j) & 1) {
                const int k0 = it.pos[j] / rfX, k1 = it.pos[j] - k0 * rfX;
                int& o = owner[(size_t)k1 * fY + k0];
                if (o >= 0) return "internal: bin written twice";
                o = (int)i * 4 + j;
            }
    }
    for (size_t c = 0; c < gt.chunks.size(); ++c)
        std::fill_n(chunk_of.begin() + gt.chunks[c].item_base, gt.chunks[c].n_items, (int)c);
    for (int k0 = 0; k0 < fY; ++k0) row[k0] = (k0 % rY) * N + k0 / rY;
    gt.wpos.assign(gt.items.size() * 4, 0xffff);
    gt.colidx.assign((size_t)fY * rfX, 0);
    std::vector<int> used(gt.chunks.size(), 0);
    for (int k1 = 0; k1 < rfX; ++k1)
        for (int k0 = 0; k0 < fY; ++k0) {
            const int o = owner[(size_t)k1 * fY + k0];
            if (o < 0) return "internal: bin not covered";
            const int c = chunk_of[o >> 2], q = used[c]++;
            gt.wpos[o] = (unsigned short)q;
            gt.colidx[(size_t)k1 * fY + row[k0]] = (int)(gt.chunks[c].item_base * gt.slots + q);
        }
    return "";
}

}  // namespace flf
