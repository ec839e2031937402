// Host-side preparation of the tile kernels (see fvmr_tiles.h).
//
// A tile is a run of consecutive device cells.  Its work-group needs, besides the tile
// cells T, the first halo ring H1 (cells across a face of T, periodic partners included:
// their limited gradients enter the face fluxes of T) and the second ring H2 (cells across
// a face of H1: their states enter the gradients of H1).  Faces are listed in the order
// faces of T (the fluxes the tile evaluates), faces of H1, then the periodic partners of
// listed faces (geometry only).  Everything a tile reads is packed contiguously per tile, so
// a work-group streams its records; only the halo states are gathered.
#include "fvmr_tiles.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>

#include "fvmr_internal.h"

namespace fvmr {

namespace {

// Hilbert index of (x, y) on a 2^16 x 2^16 grid: the textbook xy -> d walk, four bits of x and y at a time.  The walk
// turns and flips the quadrants below the one it enters; both coordinates flip together, so its state is two
// bits: axes swapped, coordinates flipped.
class HilbertWalk {
public:
    HilbertWalk() {
        for (int state = 0; state < 4; state++)
            for (int xy = 0; xy < 256; xy++) {
                int swap = state & 1, flip = state >> 1, d = 0;
                for (int b = 3; b >= 0; b--) {
                    const int x = (xy >> (4 + b)) & 1, y = (xy >> b) & 1;
                    const int rx = (swap ? y : x) ^ flip, ry = (swap ? x : y) ^ flip;
                    d = (d << 2) | ((3 * rx) ^ ry);
                    if (!ry) {
                        flip ^= rx;
                        swap ^= 1;
                    }
                }
                step_[state][xy] = (uint16_t)(d << 2 | flip << 1 | swap);
            }
    }
    uint32_t index(uint32_t x, uint32_t y) const {
        uint32_t d = 0, state = 0;
        for (int b = 12; b >= 0; b -= 4) {
            const uint32_t q = step_[state][((x >> b) & 15u) << 4 | ((y >> b) & 15u)];
            d = d << 8 | q >> 2;
            state = q & 3u;
        }
        return d;
    }

private:
    uint16_t step_[4][256];
};

bool same_bits(double a, double b) { return std::memcmp(&a, &b, sizeof(double)) == 0; }

// Green-Gauss weight g_C = |r_F - r_f| / max(|r_F - r_C|, EPSILON) of cell c across edge e to
// cell o, the neighbour's centroid shifted by the periodic translation on periodic faces
// (GradientGreenGaussKernel, FVMR/src/space/gradient/GradientGPU.cu:223-425); 0.5 without a
// cell across.
double gg_weight(const TileInput &in, int c, int e, int o, bool periodic) {
    if (o < 0) return 0.5;
    const double fx = in.mx[e], fy = in.my[e];
    double Fx = in.cx[o], Fy = in.cy[o];
    const int pe = in.edge[e].pair;
    if (periodic && pe >= 0) {
        Fx += fx - in.mx[pe];
        Fy += fy - in.my[pe];
    }
    const double ax = fx - Fx, ay = fy - Fy, bx = in.cx[c] - Fx, by = in.cy[c] - Fy;
    const double dFf = std::sqrt(ax * ax + ay * ay);
    double dFC = std::sqrt(bx * bx + by * by);
    if (dFC < kEPS) dFC = kEPS;
    return dFf / dFC;
}

// The nodes of cell c in the order of its slots: slot j joins v[j] and v[j + 1].  turned[j]: the edge's normal
// times the cell's sign (out of the cell) is (-dy, dx), not (dy, -dx), of the step v[j] -> v[j + 1].  False
// when the three edges do not join the cell's three nodes.
bool slot_nodes(const TileInput &in, int c, int v[3], int turned[3]) {
    int a[3], b[3];
    for (int j = 0; j < 3; j++) {
        const int x = in.cslot[(size_t)j * in.nc + c].x, e = x & ((1 << 28) - 1);
        a[j] = in.en0[e];
        b[j] = in.en1[e];
        if (x & (1 << 30)) std::swap(a[j], b[j]);   // the cell is R: seen from it the edge runs the other way
    }
    v[1] = (b[0] == a[1] || b[0] == b[1]) ? b[0] : a[0];
    v[0] = (v[1] == b[0]) ? a[0] : b[0];
    v[2] = (a[1] == v[1]) ? b[1] : a[1];
    for (int j = 0; j < 3; j++) {
        const int p = v[j], q = v[(j + 1) % 3];
        if (a[j] == p && b[j] == q) turned[j] = 0;
        else if (a[j] == q && b[j] == p) turned[j] = 1;
        else return false;
        bool mine = false;
        for (int k = 0; k < 3; k++) mine = mine || in.cnode[(size_t)k * in.nc + c] == p;
        if (!mine) return false;
    }
    return true;
}

}  // namespace

std::vector<int> hilbert_order(int nc, const double *cx, const double *cy) {
    double x0 = INFINITY, x1 = -INFINITY, y0 = INFINITY, y1 = -INFINITY;
    for (int c = 0; c < nc; c++) {
        x0 = std::min(x0, cx[c]); x1 = std::max(x1, cx[c]);
        y0 = std::min(y0, cy[c]); y1 = std::max(y1, cy[c]);
    }
    constexpr int order = 16;   // HilbertWalk's
    static const HilbertWalk walk;
    const double span = std::max(std::max(x1 - x0, y1 - y0), 1e-300);
    const double scale = ((1u << order) - 1) / span;
    struct Key {
        uint32_t d;
        int c;
    };
    std::vector<Key> key(nc), next(nc);
    for (int c = 0; c < nc; c++) {
        const uint32_t ix = (uint32_t)std::min<double>((cx[c] - x0) * scale, (1u << order) - 1);
        const uint32_t iy = (uint32_t)std::min<double>((cy[c] - y0) * scale, (1u << order) - 1);
        key[c] = {walk.index(ix, iy), c};
    }
    // by 11 bits at a time, each pass stable (a comparison sort takes 2.5 times as long at 393,216 cells)
    constexpr int kBits = 11;
    for (int shift = 0; shift < 2 * order; shift += kBits) {
        size_t at[1 << kBits] = {0};
        for (const Key &k : key) at[(k.d >> shift) & ((1u << kBits) - 1)]++;
        size_t sum = 0;
        for (size_t &n : at) {
            const size_t m = n;
            n = sum;
            sum += m;
        }
        for (const Key &k : key) next[at[(k.d >> shift) & ((1u << kBits) - 1)]++] = k;
        key.swap(next);
    }
    std::vector<int> order_out(nc);
    for (int i = 0; i < nc; i++) order_out[i] = key[i].c;
    return order_out;
}

void group_tiles(int n, const int *nbr, int cells, int gcells, int gmost, int ffaces, std::vector<int> &order,
                 std::vector<int> &sizes) {
    std::vector<int> tile(n, -1);                    // tile of a cell
    std::vector<int> seen(n, -1);                    // last tile that has met the cell, as cell or halo
    std::vector<int> start{0}, member;               // tile t: member[start[t]] .. member[start[t + 1]]
    member.reserve(n);
    std::vector<int> seeds, notch, front;            // cells beside finished tiles; growth queues
    size_t seed_head = 0;
    int next = 0;
    const int grow = std::max(1, cells - 1);         // the rest of the room is for cells left alone
    while ((int)member.size() < n) {
        const int t = (int)start.size() - 1;
        // the oldest cell beside a finished tile, so that tiles fill the mesh as a front, else the next free one
        int seed = -1;
        while (seed < 0 && seed_head < seeds.size()) {
            const int c = seeds[seed_head++];
            if (tile[c] < 0) seed = c;
        }
        if (seed < 0) {
            while (tile[next] >= 0) next++;
            seed = next;
        }
        const size_t first = member.size();
        int halo = 0, bfaces = 0;                    // first-ring cells, faces with one side in the tile
        notch.clear();
        front.clear();
        size_t front_head = 0;
        auto add = [&](int c) {
            tile[c] = t;
            member.push_back(c);
            if (seen[c] == t) halo--;
            seen[c] = t;
            for (int j = 0; j < 3; j++) {
                const int o = nbr[3 * (size_t)c + j];
                if (o < 0 || tile[o] != t) bfaces++;
                else if (o != c) bfaces--;
                if (o < 0 || tile[o] == t) continue;
                const bool again = seen[o] == t;
                if (!again) {
                    seen[o] = t;
                    halo++;
                }
                if (tile[o] < 0) (again ? notch : front).push_back(o);   // a second face in the tile: fill it first
            }
        };
        auto full = [&]() {
            const int s = (int)(member.size() - first);
            return s >= grow || s + halo + 2 > gcells || (3 * s + bfaces) / 2 + 3 > ffaces;
        };
        add(seed);
        while (!full()) {
            int c = -1;
            while (c < 0 && !notch.empty()) {
                if (tile[notch.back()] < 0) c = notch.back();
                notch.pop_back();
            }
            while (c < 0 && front_head < front.size()) {
                if (tile[front[front_head]] < 0) c = front[front_head];
                front_head++;
            }
            if (c < 0) break;
            add(c);
        }
        // cells whose neighbours are all in tiles would become tiles of their own
        for (size_t k = first; k < member.size(); k++)
            for (int j = 0; j < 3; j++) {
                const int o = nbr[3 * (size_t)member[k] + j];
                const int s = (int)(member.size() - first);
                if (o < 0 || tile[o] >= 0 || s >= cells || s + halo + 2 > gmost || (3 * s + bfaces) / 2 + 3 > ffaces) continue;
                bool alone = true;
                for (int q = 0; q < 3; q++) {
                    const int r = nbr[3 * (size_t)o + q];
                    alone = alone && (r < 0 || r == o || tile[r] >= 0);
                }
                if (alone) add(o);
            }
        for (size_t k = first; k < member.size(); k++)
            for (int j = 0; j < 3; j++) {
                const int o = nbr[3 * (size_t)member[k] + j];
                if (o >= 0 && tile[o] < 0) seeds.push_back(o);
            }
        std::sort(member.begin() + first, member.end());
        start.push_back((int)member.size());
    }
    // the tiles along the numbering of their middle cells
    std::vector<std::pair<int, int>> key(start.size() - 1);
    for (size_t t = 0; t + 1 < start.size(); t++) key[t] = {member[(start[t] + start[t + 1]) / 2], (int)t};
    std::sort(key.begin(), key.end());
    order.clear();
    order.reserve(n);
    sizes.clear();
    for (auto &k : key) {
        order.insert(order.end(), member.begin() + start[k.second], member.begin() + start[k.second + 1]);
        sizes.push_back(start[k.second + 1] - start[k.second]);
    }
}

bool standard_geometry(const fvmr_mesh_soa *m, const char **why) {
    const double *X = m->node_xy[0], *Y = m->node_xy[1];
    for (int c = 0; c < m->num_element; c++) {
        double sx = 0.0, sy = 0.0;
        for (int j = 0; j < 3; j++) {
            sx += X[m->element_nodes[j][c]];
            sy += Y[m->element_nodes[j][c]];
        }
        if (!same_bits(sx / 3.0, m->element_xy[0][c]) || !same_bits(sy / 3.0, m->element_xy[1][c])) {
            *why = "element centroids are not (x0+x1+x2)/3 of the node coordinates";
            return false;
        }
    }
    for (int e = 0; e < m->num_edge; e++) {
        const int a = m->edge_nodes[0][e], b = m->edge_nodes[1][e];
        const double len = m->edge_length[e];
        if (!same_bits((double)(float)len, len) || !(len > 0.0)) {
            *why = "edge lengths are not positive float values";
            return false;
        }
        if (!same_bits((X[a] + X[b]) / 2.0, m->edge_xy[0][e]) || !same_bits((Y[a] + Y[b]) / 2.0, m->edge_xy[1][e])) {
            *why = "edge midpoints are not (xa+xb)/2";
            return false;
        }
        const double dx = X[b] - X[a], dy = Y[b] - Y[a];
        if (!same_bits(dy / len, m->edge_normal[0][e]) || !same_bits(-dx / len, m->edge_normal[1][e])) {
            *why = "edge normals are not (dy,-dx)/length";
            return false;
        }
    }
    return true;
}

int build_tiles(const TileInput &in, const TileCaps &caps, TileMesh &out) {
    const int nc = in.nc, nf = in.nf;
    if (caps.cells < 1 || caps.gcells < 8 || caps.lcells < 16 || caps.nodes < 16 || caps.faces < 16 || caps.ffaces < 4 ||
        caps.lcells > kLocalNone || caps.nodes > kLocalNone || caps.faces > kLocalNone)
        return set_error(FVMR_ERR_INVALID_ARG, "bad tile capacities");
    for (int e = 0; e < nf; e++) {
        const int t = in.edge[e].type;
        if (t != -1 && (t <= kBcBase || t - kBcBase > 127))
            return set_error(FVMR_ERR_UNSUPPORTED, "boundary type outside the tile kernels' code range");
    }
    out = TileMesh();
    out.dtface.assign(nc, 0);
    // room for tiles of the usual halo (no page is touched before it is written)
    out.halo.reserve(nc);
    out.nxy.reserve(2 * (size_t)nc);
    out.lnodes.reserve(2 * (size_t)nc);
    out.lcxy.reserve(4 * (size_t)nc);
    out.gslot.reserve(4 * (size_t)nc + nc / 2);
    out.gcoef.reserve(6 * (size_t)nc);
    out.face.reserve(7 * (size_t)nc);
    out.fnrm.reserve(5 * (size_t)nc);
    auto grow = [](auto &v, size_t n) {
        v.resize(v.size() + n);
        return v.data() + v.size() - n;
    };
    // stamps: lid valid when lst == current tile
    std::vector<int> lst(nc, -1), lid(nc, 0), fst(nf, -1), fid(nf, 0);
    int nv = 0;
    for (int c = 0; c < 3 * nc; c++) nv = std::max(nv, in.cnode[c] + 1);
    for (int e = 0; e < nf; e++) nv = std::max(nv, std::max(in.en0[e], in.en1[e]) + 1);
    std::vector<int> nst(nv, -1), nid(nv, 0);
    std::vector<int> cells, faces, nodes;
    // what every tile that holds a cell packs of it
    struct Cell {
        int v[3], turned[3], last;
        double gw[3];
    };
    std::vector<Cell> rec(nc);
    for (int c = 0; c < nc && out.joined; c++) out.joined = slot_nodes(in, c, rec[c].v, rec[c].turned);
    for (int c = 0; c < nc; c++) {
        if (!out.joined)   // the vertices as they are
            for (int j = 0; j < 3; j++) {
                rec[c].v[j] = in.cnode[(size_t)j * nc + c];
                rec[c].turned[j] = 0;
            }
        rec[c].last = rec[c].v[2] == in.cnode[2 * (size_t)nc + c] ? 0 : (rec[c].v[1] == in.cnode[2 * (size_t)nc + c] ? 1 : 2);
        for (int j = 0; j < 3; j++) {
            const TileSlot sl = in.cslot[(size_t)j * nc + c];
            rec[c].gw[j] = gg_weight(in, c, sl.x & ((1 << 28) - 1), sl.y, (sl.x & (1 << 28)) != 0);
        }
    }
    int stamp = 0;

    // Builds the sets of the candidate tile [c0, c0+s); false when a capacity is exceeded.
    auto try_tile = [&](int c0, int s, int &nG, int &nFF) -> bool {
        stamp++;
        cells.clear(); faces.clear(); nodes.clear();
        auto add_cell = [&](int c) {
            if (lst[c] == stamp) return;
            lst[c] = stamp; lid[c] = (int)cells.size(); cells.push_back(c);
        };
        auto add_face = [&](int e) {
            if (fst[e] == stamp) return;
            fst[e] = stamp; fid[e] = (int)faces.size(); faces.push_back(e);
        };
        auto add_node = [&](int v) {
            if (nst[v] == stamp) return;
            nst[v] = stamp; nid[v] = (int)nodes.size(); nodes.push_back(v);
        };
        for (int i = 0; i < s; i++) add_cell(c0 + i);
        for (int i = 0; i < s; i++)
            for (int j = 0; j < 3; j++) {
                const int o = in.cslot[(size_t)j * nc + c0 + i].y;
                if (o >= 0) add_cell(o);
            }
        nG = (int)cells.size();
        if (nG > caps.gcells) return false;
        for (int i = s; i < nG; i++)
            for (int j = 0; j < 3; j++) {
                const int o = in.cslot[(size_t)j * nc + cells[i]].y;
                if (o >= 0) add_cell(o);
            }
        if ((int)cells.size() > caps.lcells) return false;
        for (int i = 0; i < s; i++)
            for (int j = 0; j < 3; j++) add_face(in.cslot[(size_t)j * nc + c0 + i].x & ((1 << 28) - 1));
        nFF = (int)faces.size();
        if (nFF > caps.ffaces) return false;
        for (int i = s; i < nG; i++)
            for (int j = 0; j < 3; j++) add_face(in.cslot[(size_t)j * nc + cells[i]].x & ((1 << 28) - 1));
        for (size_t k = 0; k < faces.size(); k++) {
            const int pe = in.edge[faces[k]].pair;
            if (pe >= 0) add_face(pe);
            if ((int)faces.size() > caps.faces) return false;
        }
        if ((int)faces.size() > caps.faces) return false;
        for (int c : cells)
            for (int j = 0; j < 3; j++) add_node(in.cnode[(size_t)j * nc + c]);
        for (int e : faces) { add_node(in.en0[e]); add_node(in.en1[e]); }
        return (int)nodes.size() <= caps.nodes;
    };

    out.case_tile_begin.assign(1, 0);
    int cs = 0;
    size_t want = 0;
    int want_end = 0;   // end of the wanted tile that c0 is in
    for (int c0 = 0; c0 < nc;) {
        while (cs + 1 < in.ncases && c0 >= in.case_begin[cs + 1]) {
            cs++;
            out.case_tile_begin.push_back(out.ntiles);
        }
        const int case_end = (cs + 1 < in.ncases) ? in.case_begin[cs + 1] : nc;
        int s = std::min(caps.cells, case_end - c0), nG = 0, nFF = 0;
        if (in.sizes) {
            while (want_end <= c0 && want < in.sizes->size()) want_end += (*in.sizes)[want++];
            if (want_end > c0) s = std::min(s, want_end - c0);
        }
        while (!try_tile(c0, s, nG, nFF)) {
            if (s == 1) return set_error(FVMR_ERR_UNSUPPORTED, "one cell and its halo exceed the tile capacity");
            s = std::max(1, s - std::max(1, s / 8));
        }
        const int nL = (int)cells.size(), nF = (int)faces.size(), nN = (int)nodes.size();
        const int info[kTileInfo] = {c0, s, nG, nL, nN, nF, nFF,
                                     (int)out.halo.size(), (int)(out.nxy.size() / 2), (int)(out.face.size() / 3),
                                     (int)out.lnodes.size(), (int)(out.gcoef.size() / 4), cs};
        out.info.insert(out.info.end(), info, info + kTileInfo);
        out.halo.insert(out.halo.end(), cells.begin() + s, cells.end());
        double *nxy = grow(out.nxy, 2 * (size_t)nN);
        for (int k = 0; k < nN; k++) {
            nxy[2 * k] = in.node_x[nodes[k]];
            nxy[2 * k + 1] = in.node_y[nodes[k]];
        }
        double *lcxy = grow(out.lcxy, 2 * (size_t)nL);
        int *lnodes = grow(out.lnodes, nL);
        for (int i = 0; i < nL; i++) {
            const int c = cells[i];
            lcxy[2 * i] = in.cx[c];
            lcxy[2 * i + 1] = in.cy[c];
            unsigned w = (unsigned)rec[c].last << kLnLastShift;
            for (int j = 0; j < 3; j++) w |= (unsigned)nid[rec[c].v[j]] << (kLocalBits * j);
            lnodes[i] = (int)w;
        }
        int *gslot = grow(out.gslot, 3 * (size_t)nG);
        double *gcoef = grow(out.gcoef, 4 * (size_t)nG);
        for (int i = 0; i < nG; i++) {
            const int c = cells[i];
            int fw = 0;
            for (int j = 0; j < 3; j++) {
                const int x = in.cslot[(size_t)j * nc + c].x, o = in.cslot[(size_t)j * nc + c].y;
                const int e = x & ((1 << 28) - 1);
                int w = fid[e] | ((o >= 0 ? lid[o] : kLocalNone) << kGsOutShift);
                fw |= fid[e] << (kLocalBits * j);
                if (x & (1 << 30)) w |= kGsIsR;
                if (x & (1 << 28)) w |= kGsPeriodic;
                if (rec[c].turned[j]) w |= kGsTurned;
                gslot[3 * i + j] = w;
                gcoef[4 * i + j] = rec[c].gw[j];
            }
            if (i < s) out.dtface[c] = fw;
            gcoef[4 * i + 3] = in.vol[c];
        }
        int *face = grow(out.face, 3 * (size_t)nF);
        double *fnrm = grow(out.fnrm, 2 * (size_t)nF);
        for (int k = 0; k < nF; k++) {
            const int e = faces[k];
            const TileEdge &ed = in.edge[e];
            const int bc = (ed.type == -1) ? 0 : ed.type - kBcBase;
            auto loc = [&](int c) { return (c >= 0 && lst[c] == stamp) ? lid[c] : kLocalNone; };
            const int pl = (ed.pair >= 0 && fst[ed.pair] == stamp) ? fid[ed.pair] : kLocalNone;
            const float lf = (float)in.elen[e];
            face[3 * k] = nid[in.en0[e]] | (nid[in.en1[e]] << kLocalBits) | (bc << kBcShift);
            face[3 * k + 1] = loc(ed.L) | (loc(ed.R) << kLocalBits) | (pl << (2 * kLocalBits));
            std::memcpy(&face[3 * k + 2], &lf, sizeof(int));
            fnrm[2 * k] = in.nx[e];
            fnrm[2 * k + 1] = in.ny[e];
        }
        out.max_nL = std::max(out.max_nL, nL); out.max_nG = std::max(out.max_nG, nG);
        out.max_nF = std::max(out.max_nF, nF); out.max_nFF = std::max(out.max_nFF, nFF);
        out.max_nN = std::max(out.max_nN, nN);
        out.sum_nL += nL; out.sum_nG += nG; out.sum_nF += nF; out.sum_nN += nN;
        out.ntiles++;
        c0 += s;
    }
    while ((int)out.case_tile_begin.size() <= in.ncases) out.case_tile_begin.push_back(out.ntiles);
    return FVMR_OK;
}

}  // namespace fvmr
