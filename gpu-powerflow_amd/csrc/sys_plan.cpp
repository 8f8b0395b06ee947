#include "sys_plan.hpp"

#include <algorithm>
#include <cstring>

namespace cupf {

namespace {
// LDS elements of a front's factors.
long long factor_elems(int fs, int K) { return (long long)K * (fs | 1) + (long long)(fs - K) * (K | 1); }

// A front is shared by the whole workgroup when its level has too few fronts
// to occupy the waves, or when it exceeds a wave's registers.
constexpr int kAloneFronts = 2;
constexpr int kWaveRows = 32;

// First-fit allocation of blocks with lifetimes [from, to] (levels).
struct Arena {
    struct Block { int off, len, from, to; };
    std::vector<Block> blocks;
    int top = 0;
    int take(int len, int from, int to) {
        std::vector<std::pair<int, int>> busy;
        for (const Block& b : blocks)
            if (b.len > 0 && b.from <= to && from <= b.to) busy.push_back({b.off, b.off + b.len});
        std::sort(busy.begin(), busy.end());
        int at = 0;
        for (const auto& r : busy) {
            if (at + len <= r.first) break;
            at = std::max(at, r.second);
        }
        blocks.push_back({at, len, from, to});
        top = std::max(top, at + len);
        return at;
    }
};
}  // namespace

SysPlan make_sys_plan(const LuPlan& P, size_t most_elems) {
    SysPlan S;
    S.n = P.n;
    S.nnz = P.nnz;
    const int F = P.num_fronts;
    if (P.max_fsz > kSysMaxRows || P.max_nc > 64 || P.n >= 0xffff || F >= 0xffff || P.num_levels >= 0xffff)
        return S;
    std::vector<int> parent(size_t(F), -1);
    for (int p = 0; p < F; ++p)
        for (int q = P.child_ptr[p]; q < P.child_ptr[p + 1]; ++q) parent[size_t(P.child_idx[q])] = p;

    std::vector<SysFront> fr(static_cast<size_t>(F));
    Arena arena;
    long long fac = 0, work = 0;
    std::vector<int> order(static_cast<size_t>(F));
    for (int p = 0; p < F; ++p) order[size_t(p)] = p;
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return P.level[a] < P.level[b]; });
    // sizes first: a system that is too large costs one pass over its fronts,
    // and the allocation below (fronts squared) ends where the blocks no longer fit
    for (int p = 0; p < F; ++p) {
        fac += factor_elems(P.fsz[p], P.nc[p]);
        work += P.fsz[p];
    }
    if (size_t(fac + work) > most_elems) return S;
    for (int p : order) {
        const int fs = P.fsz[p], K = P.nc[p], uc = fs - K;
        const int to = parent[size_t(p)] >= 0 ? P.level[parent[size_t(p)]] : P.level[p];
        fr[size_t(p)].co = arena.take(uc * uc, P.level[p], to);
        if (size_t(fac + arena.top) > most_elems) return S;
    }
    fac = work = 0;
    for (int p = 0; p < F; ++p) {
        const int fs = P.fsz[p], K = P.nc[p];
        SysFront& f = fr[size_t(p)];
        f.fo = int(fac);
        f.wo = int(work);
        fac += factor_elems(fs, K);
        work += fs;
        f.size = fs | K << 16;
        f.first = P.front_rows[P.front_ptr[p]];
        for (int k = 0; k < K; ++k)
            if (P.front_rows[P.front_ptr[p] + k] != f.first + k) return S;   // pivots lead, consecutive
        f.rows = P.front_ptr[p];
    }
    S.fac = int(fac);
    S.scratch = int(std::max<long long>(arena.top, work)) + 1;
    if (size_t(S.fac) + size_t(S.scratch) > most_elems) return S;
    const int zero = S.fac + S.scratch - 1;              // an element no block or vector uses
    if (zero >= 0xffff || P.front_ptr[F] >= 0xffff || P.gat_ptr[size_t(P.front_ptr[F])] >= 0xffff) return S;

    // additions by destination, children in child order
    std::vector<int> slices, cnt, dst, from, at;
    for (int p = 0; p < F; ++p) {
        const int fs = P.fsz[p], K = P.nc[p], uc = fs - K;
        SysFront& f = fr[size_t(p)];
        // sources of each element, by counts
        cnt.assign(size_t(fs) * fs + 1, 0);
        auto children = [&](auto add) {
            for (int q = P.child_ptr[p]; q < P.child_ptr[p + 1]; ++q) {
                const int c = P.child_idx[q], cuc = P.fsz[c] - P.nc[c];
                const int* loc = P.asm_loc.data() + P.asm_ptr[c];
                for (int a = 0; a < cuc; ++a)
                    for (int b = 0; b < cuc; ++b)
                        add(size_t(loc[a]) * fs + loc[b], S.fac + fr[size_t(c)].co + a * cuc + b);
            }
        };
        children([&](size_t e, int) { ++cnt[e + 1]; });
        dst.clear();
        for (int e = 0; e < fs * fs; ++e) {
            if (cnt[size_t(e) + 1]) dst.push_back(e);
            cnt[size_t(e) + 1] += cnt[size_t(e)];
        }
        from.resize(size_t(cnt.back()));
        at.assign(cnt.begin(), cnt.end() - 1);
        children([&](size_t e, int src) { from[size_t(at[e]++)] = src; });
        auto width_of = [&](int e) { return cnt[size_t(e) + 1] - cnt[size_t(e)]; };
        std::stable_sort(dst.begin(), dst.end(), [&](int a, int b) { return width_of(a) > width_of(b); });
        f.slice0 = int(slices.size());
        for (size_t d0 = 0; d0 < dst.size(); d0 += 16) {
            const int width = width_of(dst[d0]);
            if (width > 0xff || S.adds.size() / 16 >= (1u << kSysSliceShift)) return S;
            slices.push_back(int(unsigned(S.adds.size() / 16) | unsigned(width) << kSysSliceShift));
            for (int r = 0; r < 1 + width; ++r)
                for (size_t l = 0; l < 16; ++l) {
                    // lanes past the end repeat the last destination's work
                    const int e = dst[std::min(d0 + l, dst.size() - 1)];
                    const int i = e / fs, j = e % fs;
                    const int to = i < K ? f.fo + i * (fs | 1) + j
                                 : j < K ? f.fo + K * (fs | 1) + (i - K) * (K | 1) + j
                                         : S.fac + f.co + (i - K) * uc + (j - K);
                    S.adds.push_back(uint16_t(r == 0              ? to
                                              : r <= width_of(e) ? from[size_t(cnt[size_t(e)] + r - 1)]
                                                                 : zero));
                }
        }
        f.slices = int(slices.size()) - f.slice0;
    }
    for (int l = 0; l < 16; ++l) S.adds.push_back(uint16_t(zero));   // the kernels read a row ahead
    // solve gather: the children's work-vector elements landing on each position
    std::vector<int> gsrc(P.gat_src.size(), 0);
    {
        at.assign(P.gat_ptr.begin(), P.gat_ptr.end() - 1);
        for (int p = 0; p < F; ++p)
            for (int q = P.child_ptr[p]; q < P.child_ptr[p + 1]; ++q) {
                const int c = P.child_idx[q];
                const int* loc = P.asm_loc.data() + P.asm_ptr[c];
                for (int a = 0; a < P.fsz[c] - P.nc[c]; ++a)
                    gsrc[size_t(at[size_t(P.front_ptr[p] + loc[a])]++)] = S.fac + fr[size_t(c)].wo + P.nc[c] + a;
            }
    }

    // tasks per level: wave fronts largest first, then the quads, then shared fronts
    std::vector<int> levels;
    std::vector<uint16_t> task;
    for (int L = 0; L < P.num_levels; ++L) {
        std::vector<int> small, big;
        for (int p = 0; p < F; ++p)
            if (P.level[p] == L) (P.fsz[p] <= kSysSmallRows ? small : big).push_back(p);
        std::stable_sort(big.begin(), big.end(), [&](int a, int b) { return P.fsz[a] > P.fsz[b]; });
        std::stable_sort(small.begin(), small.end(), [&](int a, int b) { return P.nc[a] > P.nc[b]; });
        std::vector<int> wide, wave;
        for (int p : big)
            (int(big.size()) <= kAloneFronts || P.fsz[p] > kWaveRows ? wide : wave).push_back(p);
        levels.push_back(int(task.size()));
        const int quads = int(small.size() + 3) / 4;
        levels.push_back(quads);
        levels.push_back(int(wave.size()));
        levels.push_back(int(wide.size()));
        for (int p : wave) task.push_back(uint16_t(p));
        for (int q = 0; q < quads * 4; ++q)
            task.push_back(q < int(small.size()) ? uint16_t(small[size_t(q)]) : uint16_t(0xffff));
        for (int p : wide) task.push_back(uint16_t(p));
    }

    // blob: fronts, levels, slices, then the u16 lists
    S.num_fronts = F;
    S.num_levels = P.num_levels;
    S.o_level = F * int(sizeof(SysFront) / sizeof(int));
    S.o_slice = S.o_level + int(levels.size());
    const int ints = S.o_slice + int(slices.size());
    std::vector<uint16_t> lists;
    auto put = [&](const auto& v) {
        const int at = int(lists.size());
        for (auto x : v) lists.push_back(uint16_t(x));
        return at + 2 * ints;
    };
    S.o_task = put(task);
    S.o_rows = put(P.front_rows);
    S.o_gptr = put(P.gat_ptr);
    S.o_gsrc = put(gsrc);
    S.o_perm = put(P.perm);
    S.blob.assign(size_t((ints + int(lists.size() + 1) / 2 + 3) / 4 * 4), 0);
    std::memcpy(S.blob.data(), fr.data(), fr.size() * sizeof(SysFront));
    std::copy(levels.begin(), levels.end(), S.blob.begin() + S.o_level);
    std::copy(slices.begin(), slices.end(), S.blob.begin() + S.o_slice);
    std::memcpy(S.blob.data() + ints, lists.data(), lists.size() * sizeof(uint16_t));

    S.slot_pos.assign(size_t(P.nnz), -1);
    for (int p = 0; p < F; ++p) {
        const int fs = P.fsz[p], K = P.nc[p];
        for (int e = P.ent_ptr[p]; e < P.ent_ptr[p + 1]; ++e) {
            const int r = P.ent_dst[e] / fs, c = P.ent_dst[e] % fs;
            if (r >= K && c >= K) return S;              // an entry belongs to a pivot row or column
            S.slot_pos[size_t(P.ent_src[e])] =
                r < K ? fr[size_t(p)].fo + r * (fs | 1) + c
                      : fr[size_t(p)].fo + K * (fs | 1) + (r - K) * (K | 1) + c;
        }
    }
    S.ok = true;
    return S;
}

SysPlan find_sys_plan(const LuPlan& P, const Symbolic& sym, const int* rp, const int* ci, size_t most_elems) {
    // Entries of L and U off the diagonal: the least elements of the factors at
    // any cap, known without another analysis.  Fronts only grow with the cap,
    // so those of a narrower plan tell too.
    if (size_t(2 * (P.lnz - P.n)) > most_elems || (sym.cap <= kSysCap && P.max_fsz > kSysMaxRows))
        return SysPlan{};
    if (sym.cap == kSysCap) return make_sys_plan(P, most_elems);
    Symbolic at = sym;
    cut_panels(at, kSysCap);
    long long fac = 0;
    for (int p = 0; p < at.num_panels; ++p) fac += factor_elems(at.front_ptr[p + 1] - at.front_ptr[p], at.panel_ncols[p]);
    if (size_t(fac) > most_elems) return SysPlan{};
    return make_sys_plan(lower_plan(at, P.n, rp, ci), most_elems);
}

}  // namespace cupf
