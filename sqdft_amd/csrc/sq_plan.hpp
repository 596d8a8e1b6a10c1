// sq_plan.hpp -- sizes and rules behind the launches of the grouped projector
// kernels: how a batch is cut into groups, which shape and how much LDS a walk
// takes.  Plain C++ without HIP, so that the rules can be tested on the CPU.
#pragma once

#include <algorithm>
#include <cstddef>
#include <utility>
#include <vector>

namespace sqk {

constexpr int LCAP = 512;       // max images meeting one node cube
constexpr int NG = 8;           // node cubes per workgroup of the grouped projector kernels
constexpr int SLW = 10;         // LDS row of k_nlapplyg: NG projections padded to 80 B (rows
                                // r and r + 4 would share banks at 64 B)
constexpr int GLCAP = 1024;     // max images meeting the cubes of one group
constexpr int MAXIT = 500;      // Lanczos max_iter (sq.cpp:967)
constexpr size_t LDS_MAX = 160 * 1024;

// Image data that k_projs and k_projw read per image and plane, cached in LDS per group
struct ImgMeta {
    int ox, oy, oz;               // rc-box origin (unwrapped grid coordinates)
    int w, np, t, ipb;            // box side, projectors, type, first image-projector id
    long uoff;                    // offset of the image's U block in udv
};

// Visiting order of the FD nodes: bricks of up to 4x4x2 nodes, so that
// workgroups that run at the same time (consecutive batch slots) march
// overlapping cubes and share Veff, projector tables and ELL entries in the
// caches.  Each axis is cut into near-equal runs (of up to 4, 2 and 2 nodes in
// x, y and z; a brick is two y runs), so a grid side that 4 does not divide
// has no thin last brick.  The nodes of one (x run, y run, z) are consecutive:
// the up to 4x2x1 block that one projection workgroup takes.
// The host orders while the GPU waits: walking the bricks, 96^3 nodes take 2 ms
// where sorting them by key took 46 (a density step with 7^3 cubes, mixed
// precision, 455 ms in all).
struct NodeOrder {
    int n;
    std::vector<int> sx, sy, sz;   // where the runs of each axis start, and n
    std::vector<int> rx, ry, rz;   // run of each coordinate
    explicit NodeOrder(int n_) : n(n_) { runs(4, sx, rx); runs(2, sy, ry); runs(2, sz, rz); }
    void runs(int len, std::vector<int> &s, std::vector<int> &r) const
    {
        const int m = (n + len - 1) / len;
        r.resize(n);
        for (int c = 0; c <= m; ++c) s.push_back((int)((long)c * n / m));
        for (int c = 0; c < m; ++c) std::fill(r.begin() + s[c], r.begin() + s[c + 1], c);
    }
    // the nodes of the z-planes [z0, z0 + nz)
    std::vector<int> planes(int z0, int nz) const
    {
        std::vector<int> out;
        out.reserve((size_t)nz * n * n);
        const int my = (int)sy.size() - 1;
        for (size_t bz = 0; bz + 1 < sz.size(); ++bz)
            for (int by = 0; by < my; by += 2)
                for (size_t bx = 0; bx + 1 < sx.size(); ++bx)
                    for (int z = std::max(sz[bz], z0); z < std::min(sz[bz + 1], z0 + nz); ++z)
                        for (int y = sy[by]; y < sy[std::min(by + 2, my)]; ++y)
                            for (int x = sx[bx]; x < sx[bx + 1]; ++x) out.push_back((z * n + y) * n + x);
        return out;
    }
    // sort key: brick z, y, x; then z, y, x
    unsigned long key(int node) const
    {
        const int x = node % n, y = (node / n) % n, z = node / (n * n);
        const unsigned long m = (unsigned long)n + 1;
        unsigned long k = rz[z];
        for (int f : {ry[y] / 2, rx[x], z, y, x}) k = k * m + (unsigned long)f;
        return k;
    }
    // any list, repeats allowed
    void sort(std::vector<int> &nodes) const
    {
        size_t i = 1;
        for (unsigned long k = nodes.empty() ? 0 : key(nodes[0]), q; i < nodes.size(); ++i, k = q)
            if ((q = key(nodes[i])) < k) break;
        if (i >= nodes.size()) return;
        const size_t nn = (size_t)n * n * n;
        if (nodes.size() * 8 >= nn) {   // a good part of the grid: count and walk it
            std::vector<int> cnt(nn, 0);
            for (int v : nodes) ++cnt[v];
            size_t o = 0;
            for (int v : planes(0, n))
                for (int c = cnt[v]; c > 0; --c) nodes[o++] = v;
            return;
        }
        std::vector<std::pair<unsigned long, int>> k(nodes.size());
        for (size_t j = 0; j < nodes.size(); ++j) k[j] = {key(nodes[j]), nodes[j]};
        std::sort(k.begin(), k.end());
        for (size_t j = 0; j < nodes.size(); ++j) nodes[j] = k[j].second;
    }
};

// What the rules depend on: cube side, most projectors of an image, number of
// image-projectors, side of the widest rc-box.
struct ProjDims { int M, max_nproj, n_ip, w; };

// The most values by which a member's cube may start after the corner of its
// group's union: one plane, and rows and columns within (M + 3)^2 (the rule of
// make_groups, whatever order the nodes come in).
constexpr int group_pad(int M) { return M * M + 6 * M + 24; }

// Values in the resources of k_projw and k_nlapplyg: from group_pad before the
// group's first vector to past a full group's last one.  Every scalar offset below
// lies inside, that of an idle member (past the group's end or frozen) too, so that
// nothing rests on what the hardware's range check makes of one past the end.
// Lanes stay within the members' vectors by their masks: a masked lane's own
// offset lies past the range.
constexpr int group_range(int M) { return NG * M * M * M + 2 * group_pad(M); }

// Scalar offset, in values, that takes an offset inside the group's union
// (z M^2 + y M + x from its corner) to member m's vector; dx, dy, dz: the corner
// minus the start of the member's cube, pad: group_pad (M2 and M3 come from the
// caller: formed again from M they cost the FP64 Lanczos walk 6 % of its time).
constexpr int member_offset(int m, int pad, int M, int M2, int M3, int dx, int dy, int dz)
{
    return pad + m * M3 + dz * M2 + dy * M + dx;
}

// Compiled shapes of k_projw, the first that holds every group of the batch is
// taken: waves per workgroup and register slots per wave.  One workgroup fills
// a CU's LDS, so its waves are all that hides the loads: twelve, if the slots
// that their 168 VGPRs hold are enough (the Al and LiH cells), else eight with
// more slots.  Twelve against eight, us a pass: 8,192 nodes with FP64 35^3
// cubes 1265 against 1549 (Lanczos) and 895 against 1175 (Chebyshev), 4,096
// with FP32 ones 468 and 402 against 542 and 488; MFMA, 4,096 nodes with 31^3
// cubes, 875 and 862 against 1142 and 1166.  With the union columns worked out
// once per walk the twelve-wave ones take 1192, 863, 459, 358, 838 and 760.
// Eight waves help only with more slots in all: a walk that R slots in twelve waves
// do not hold has 12 R + 1 consecutive images alive, so one of eight waves needs
// 3 R / 2 + 1 slots at least.
constexpr int PROJW_RPI = 3;
struct ProjShape { int nw, R; };
constexpr ProjShape PROJR_SHAPES[3] = {{12, 4}, {8, 10}, {8, 16}};
constexpr ProjShape PROJM_SHAPES[1] = {{12, 12}};   // MFMA: two doubles per slot and lane
constexpr int PROJ_NW[2] = {12, 8};
constexpr int PR_DEPTHS = 2;    // slab depths in question on one batch at most

// How k_projw runs on vectors of ts bytes per value: on = 0 when it does not
// apply; the matrix cores for FP64 tables of several projectors.
struct ProjwUse { int on, mfma, w; };
inline ProjwUse projw_use(const ProjDims &d, size_t ts)
{
    if (d.max_nproj < 1 || d.max_nproj > 4 || d.n_ip == 0) return {0, 0, 0};
    // p channels in FP64: the matrix cores.  FP32 tables (mixed precision)
    // stay with k_projs: its VALU sums of FP32 operands ran at 1.18 ms a pass
    // on the 216-atom LiH batches against 1.67 ms (FP64 MFMAs fed by
    // conversions), while in FP64 the two tied (2.3 ms).
    if (d.max_nproj > 1 && ts == 4) return {0, 0, 0};
    const int mfma = d.max_nproj > 1;
    if (mfma ? d.w > 16 : d.w * d.w > 64 * PROJW_RPI) return {0, 0, 0};
    return {1, mfma, d.w};
}

// LDS values per plane and member of a staged block of ux x uy columns: rows
// padded to a pitch congruent to the box side modulo 32, the MFMA member
// stride to 8 (as k_projw pads them).
inline int projw_slab(const ProjwUse &pw, int ux, int uy)
{
    const int u = (ux + (((pw.w - ux) % 32) + 32) % 32) * uy;
    return pw.mfma ? u + (((8 - u) % 32) + 32) % 32 : u;
}

// k_projs' slab capacity: the union plane of a 4x4 footprint of cubes.
inline int projs_pu(int M) { return (M + 3) * (M + 3); }

// k_projw's slab capacity per plane and member: the union plane of a 4x2 block of
// cubes or one cube; without padded rows any union that make_groups forms.
inline int projw_pu(int M, const ProjwUse &pw, bool pad = true)
{
    if (!pad) return projs_pu(M) + (pw.mfma ? 31 : 0);
    return std::max(projw_slab(pw, M + 3, M + 1), projw_slab(pw, M, M));
}

// LDS bytes of a list of image data
inline size_t images_lds(int images) { return ((size_t)std::max(images, 1) * sizeof(ImgMeta) + 15) / 16 * 16; }

// LDS bytes of a table of a union's columns
inline size_t columns_lds(int M)
{
    return (std::max((size_t)(M + 3) * (M + 3), (size_t)(M + 7) * M) * 4 + 15) / 16 * 16;
}

// LDS bytes of k_projw beside the slab: image data and union columns.
inline size_t projw_head(int M, int images) { return images_lds(images) + columns_lds(M); }

// Depths (planes per slab) that k_projw may walk in, the preferred one first.
// VALU: one FP64 or two FP32 planes (a deeper slab keeps more images alive than the
// slots of twelve waves: 17^3 cubes with three planes took 269 us a pass with ten
// slots in eight waves against 81).  MFMA, whose slots are small: about four load
// rounds of a workgroup between two barriers, at most eight planes, as far as the
// LDS holds them beside a list of 256 images (25^3 cubes, two planes: 373 against
// 496 us a pass); or one plane, which never keeps more images alive than several do,
// where a deep slab takes more slots than there are (4,096 nodes with 21^3 cubes and
// 418 images a group: 537 us a pass, 675 in k_projs).  A list too long for the deep
// slab alone is shared out instead (29^3 cubes, 402 images: 752 against 855 us).
struct ProjwDepths { int n, sz[PR_DEPTHS]; };
inline ProjwDepths projw_depths(int M, const ProjwUse &pw, size_t ts)
{
    if (!pw.on) return {0, {0, 0}};
    if (!pw.mfma) return {1, {ts == 4 ? 2 : 1, 0}};
    const size_t plane = (size_t)projw_pu(M, pw) * NG * ts, head = projw_head(M, 256);
    const int lds = plane + head <= LDS_MAX ? (int)((LDS_MAX - head) / plane) : 1;
    const int deep = std::max(1, std::min({8, lds, 3072 / ((M + 3) * (M + 1))}));
    return {deep > 1 ? 2 : 1, {deep, 1}};
}

// Cuts B slots into groups of up to NG consecutive ones whose cubes the
// staged projection kernels can walk together: the union plane fits the slab
// capacity of every kernel that may run on the batch (vectors of ts[0 .. nts)
// bytes per value), and the cubes are at most one plane apart in z.  A run ends
// where the next node is too far away (a brick's edge, a gap in the caller's
// list): walking such members one after the other in one workgroup, as unions
// that do not fit would need, is several times slower: with runs of 8 slots cut
// anywhere, a density step on a 15^3 LiH grid (25^3 cubes) took 534 ms and on a
// 10^3 Al grid (17^3) 44.6 ms, against 155 and 15.2 ms.
inline std::vector<int> make_groups(const ProjDims &dm, int n, const size_t *ts, int nts, const int *nodes, int B)
{
    const int M = dm.M;
    std::vector<ProjwUse> use;
    for (int i = 0; i < nts; ++i)
        if (projw_use(dm, ts[i]).on) use.push_back(projw_use(dm, ts[i]));
    auto fits = [&](int dx, int dy, int dz) {
        if (dz > 1 || (M + dx) * (M + dy) > projs_pu(M)) return false;
        for (const ProjwUse &pw : use)
            if (projw_slab(pw, M + dx, M + dy) > projw_pu(M, pw)) return false;
        return true;
    };
    std::vector<int> gst{0};
    int lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0}, r[3] = {0, 0, 0};
    for (int b = 0; b < B; ++b) {
        // the next node of a row needs no division (they are most of the work)
        if (b && nodes[b] == nodes[b - 1] + 1 && r[0] + 1 < n) {
            ++r[0];
        } else {
            r[0] = nodes[b] % n; r[1] = (nodes[b] / n) % n; r[2] = nodes[b] / (n * n);
        }
        const int cnt = b - gst.back();
        int l[3], h[3];
        for (int d = 0; d < 3; ++d) {
            l[d] = cnt ? std::min(lo[d], r[d]) : r[d];
            h[d] = cnt ? std::max(hi[d], r[d]) : r[d];
        }
        if (cnt && (cnt == NG || !fits(h[0] - l[0], h[1] - l[1], h[2] - l[2]))) {
            gst.push_back(b);
            for (int d = 0; d < 3; ++d) l[d] = h[d] = r[d];
        }
        for (int d = 0; d < 3; ++d) { lo[d] = l[d]; hi[d] = h[d]; }
    }
    gst.push_back(B);
    return gst;
}

// Workgroups that share the images of a group in k_projw.  A workgroup fills a
// CU, so ng groups take ceil(ng / 256) rounds.  Half of a group's images,
// consecutive in z, take 0.6 of a whole walk (they reach about three quarters of
// its planes), a quarter 0.52: shares pay where they fill CUs that would idle.
// us a pass with 1, 2 and 4 workgroups: a few nodes 63, 45, 36; 64 groups of
// 17^3 cubes 25, 21, 19; about 150 of them 74, 88, 96; 364 of 25^3 LiH cubes 418,
// 384, 466; 480 of them 385, 453, 565.
inline int projw_split(int ng)
{
    int best = 1;
    double t = 1e30;
    const double cost[3] = {1.0, 0.6, 0.52};
    for (int i = 0; i < 3; ++i) {
        const double ti = (((long)ng << i) + 255) / 256 * cost[i];
        if (ti < t) { t = ti; best = 1 << i; }
    }
    return best;
}

// How k_projw walks a batch: compiled shape (-1: not at all), planes per slab,
// workgroups that a group's images are shared out to at least, padded rows, LDS
// bytes of one workgroup.
struct ProjwPlan { int shape = -1, sz = 0, shares = 1, pad = 1; size_t lds = 0; };

// need[k]: register slots that any group's walk in the k-th depth takes with
// PROJ_NW[0] and PROJ_NW[1] waves; gl_max: images of the longest group list.  The
// image data must fit beside the slab and the column table; where only the table is
// too much, the images are shared out (a share holds its own images' data alone), or
// the rows go unpadded.  The sums are the same in every plan, so batches stay
// bitwise alike.
inline ProjwPlan projw_plan(int M, const ProjwUse &pw, size_t ts, int gl_max, const int (*need)[2])
{
    const ProjwDepths dep = projw_depths(M, pw, ts);
    const ProjShape *sh = pw.mfma ? PROJM_SHAPES : PROJR_SHAPES;
    const int nsh = pw.mfma ? 1 : 3;
    int shape[PR_DEPTHS] = {-1, -1};
    for (int k = 0; k < dep.n; ++k)
        for (int i = 0; i < nsh && shape[k] < 0; ++i)
            if (need[k][sh[i].nw == PROJ_NW[1]] <= sh[i].R) shape[k] = i;
    auto slab = [&](int sz, bool pad) { return (size_t)projw_pu(M, pw, pad) * NG * ts * sz; };
    for (int k = 0; k < dep.n; ++k) {
        const bool room = images_lds(gl_max) + slab(dep.sz[k], true) <= LDS_MAX;   // but for the table
        if (shape[k] < 0 || !room) continue;
        for (int pad : {1, 0})
            for (int shares : {1, 2, 4}) {
                const size_t lds = projw_head(M, (gl_max + shares - 1) / shares) + slab(dep.sz[k], pad);
                if (lds <= LDS_MAX) return {shape[k], dep.sz[k], shares, pad, lds};
            }
    }
    return {};
}

// k_projs: planes per slab (at most `deep`) and workgroups that share a group's
// images, as few as hold the image data beside the deepest slab; sz 0: does not fit.
struct ProjsPlan { int sz, shares; size_t lds; };
inline ProjsPlan projs_plan(int M, size_t ts, int deep, int gl_max)
{
    for (int shares : {1, 2, 4})
        for (int sz : {deep, deep / 2, 1}) {
            const size_t lds = images_lds((gl_max + shares - 1) / shares) + (size_t)projs_pu(M) * NG * ts * sz;
            if (lds <= LDS_MAX) return {sz, shares, lds};
        }
    return {0, 0, 0};
}

// LDS bytes of one k_nlapplyg workgroup: loc table, NG values per row and, where
// they fit as well, the union columns (else worked out point by point).
struct NlapplyPlan { bool fits, columns; size_t lds; };
inline NlapplyPlan nlapply_plan(const ProjDims &d, int gl_max)
{
    const size_t base = ((size_t)std::max(d.n_ip, 1) * 4 + 15) / 16 * 16 +
                        (size_t)std::max(gl_max * d.max_nproj, 1) * SLW * sizeof(double);
    const size_t all = base + std::max((size_t)(d.M + 3) * (d.M + 3), (size_t)(d.M + 7) * d.M) * 4;
    if (all <= LDS_MAX) return {true, true, all};
    return {base <= LDS_MAX, false, base};
}

// Workgroups that share a group's planes in k_nlapplyg, with at least four points a
// thread each.  Three of them share a CU: about eight rounds for tables of one
// projector, so that the last one costs little, four for several, whose rows every
// share fills again.  us a pass with 8 and 4 rounds: 8,192 nodes with 35^3 Al cubes
// 735 and 775; with 31^3 LiH cubes 912 and 858 (FP32 623 and 590), 4,096 of them 388
// and 373.
inline int nlapply_split(const ProjDims &d, int ng)
{
    const int pts = (d.M + 3) * (d.M + 1) * d.M, wgs = d.max_nproj > 1 ? 3072 : 6144;
    return std::max(1, std::min(wgs / std::max(ng, 1), pts / (4 * 512)));
}

// Device bytes that a batch holds per node: nvec + 3 vectors of rs bytes per value
// (the two Lanczos pairs and the nonlocal term, and what a pass adds), the
// projections, the Lanczos tridiagonals with their scratch, and scalars ...
inline size_t batch_node_bytes(const ProjDims &d, size_t rs, int nvec)
{
    return (nvec + 3) * (size_t)d.M * d.M * d.M * rs + (size_t)std::max(d.n_ip, 1) * 8 + 4 * (MAXIT + 2) * 8 + 256;
}

// ... and of image lists at most: those of a group, which may hold one node where
// the nodes are far apart, and a node's own (the forces).
constexpr size_t batch_list_bytes(bool node_lists)
{
    return (GLCAP + 2) * sizeof(int) + (node_lists ? (LCAP + 1) * sizeof(int) : 0);
}

// Per-call buffers of the allocation-free H v of nb nodes in ng groups, in
// bytes: vectors of rs bytes per value, FP32 copies of the input, the output and
// Veff (nn values) where mixed.
struct NoallocSizes {
    size_t node_list, gst, glist, glist_cnt, flags, s, NLv, X, Y, veff;
    static constexpr size_t round(size_t b) { return (b + 255) / 256 * 256; }
    NoallocSizes(const ProjDims &d, int nb, size_t ng, size_t rs, bool mixed, size_t nn)
    {
        const size_t len = (size_t)nb * d.M * d.M * d.M;
        node_list = nb * sizeof(int);
        gst = (ng + 1) * sizeof(int);
        glist = ng * GLCAP * sizeof(int);
        glist_cnt = ng * sizeof(int);
        flags = 16 * sizeof(int);
        s = (size_t)nb * std::max(d.n_ip, 1) * sizeof(double);
        NLv = len * rs;
        X = Y = mixed ? len * rs : 0;
        veff = mixed ? nn * rs : 0;
    }
    // what they take, each rounded to 256 bytes
    size_t total() const
    {
        size_t t = 0;
        for (size_t b : {node_list, gst, glist, glist_cnt, flags, s, NLv, X, Y, veff}) t += round(b);
        return t;
    }
};

// Scratch bytes by which nb nodes are taken or refused (the limit that callers
// see): full groups, and LCAP + 1 ints a node, room for lists of its own that this
// path does not build and that lists of groups with fewer nodes may take.
inline size_t noalloc_limit(const ProjDims &d, int nb, size_t rs, bool mixed, size_t nn)
{
    const NoallocSizes z(d, nb, (size_t)(nb + NG - 1) / NG, rs, mixed, nn);
    return z.total() - z.round(z.gst) + z.round((size_t)nb * LCAP * sizeof(int)) + z.round((size_t)nb * sizeof(int));
}

}  // namespace sqk
