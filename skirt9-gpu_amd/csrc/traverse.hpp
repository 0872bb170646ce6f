// Device-side path segment generators for the MI355X engine.
//
// The generators reproduce SKIRT's PathSegmentGenerator state machine bit for bit in FP64
// (this file is compiled with -ffp-contract=off so no multiply-add is fused):
//   moveInside          PathSegmentGenerator.cpp:11-112
//   Cartesian next()    CartesianSpatialGrid.cpp:77-153
//   octree next()       TreeSpatialGrid.cpp:143-228, TreeNode.cpp:66-76/103-112, OctTreeNode.cpp:37-42
//   Voronoi next()      VoronoiMeshSnapshot.cpp:1094-1213, cellIndex :1037-1071
//   tetra next()        TetraMeshSpatialGrid.cpp:697-820, findEnteringFace :87-108, contains :110-133,
//                       cellIndex :615-624
// One lane owns one path, or four lanes of a Voronoi path's; the generator state lives in registers.
#pragma once

#include <hip/hip_runtime.h>
#include <cfloat>
#include <cstddef>
#include <cstdint>

namespace skg
{
    enum GridType : int
    {
        kCartesian = 0,
        kOctree = 1,
        kVoronoi = 2,
        kTetra = 3
    };

    // Voronoi cell record (indexed by cell, for the search of a position's cell): the site and the
    // cell's run in the entry table.
    struct alignas(32) VorCell
    {
        double x, y, z;
        int32_t run;
        int32_t pad;
    };
    static_assert(sizeof(VorCell) == 32, "Voronoi cell record must be 32 bytes");

    // The entry table holds one run of 16-byte slots per cell, at a multiple of four slots: the
    // cell's head (three slots), then one entry per neighbour, padded with NaN (which the exit
    // search rejects) to at least kVorPad.  A crossing reads the run of the
    // cell that it enters and nothing else, all of it in flight at once.
    struct alignas(16) VorHead
    {
        double x, y, z;   // the site
        double dens;
        int32_t count;    // neighbours
        int32_t cell;
        float r2, r1;     // the largest squared length and 1-norm of the neighbours' offsets
    };
    static_assert(sizeof(VorHead) == 48 && offsetof(VorHead, dens) == 24 && offsetof(VorHead, count) == 32,
                  "head layout that VorRun reads");
    // The neighbour's site relative to the cell's, in units of the domain's largest side and rounded
    // to FP32, and the neighbour's run (its first slot).  Domain walls have ids -1..-6 (xmin, xmax,
    // ymin, ymax, zmin, zmax) and the site's mirror image as their site.  The exit search bounds
    // every neighbour's exit distance in FP32 and computes the FP64 distance of the only one that
    // can be the smallest: 16 bytes instead of 32 per neighbour, and one FP64 division per crossing.
    struct alignas(16) VorNb
    {
        float x, y, z;
        int32_t id;
    };
    static_assert(sizeof(VorNb) == 16, "Voronoi neighbour entry must be 16 bytes");
    constexpr int kVorPad = 12;  // entries every run has room for
    // entries a lane has in flight where L lanes share a path (400 000 sites, 2^18 packets, L = 1 with
    // 6 / 8 / 10 / 12: 40.8 / 39.6 / 40.1 / 43.0 ms)
    template<int L> constexpr int kVorAhead = L == 4 ? 5 : 8;
    constexpr int kVorSlack = 32;  // slots behind the last run that may be read (and are not used)
    // relative error allowed to the FP32 bounds: the offsets, the position and five operations are
    // each rounded to within 2^-24 of products that (n.n + w.w) or |n| |k| bound, in sum below 2^-21
    constexpr float kVorEps = 0x1p-19f;
    // offsets shorter than this (of the largest of the domain's side and its coordinates) are stored
    // as zero: the FP64 distances themselves are less exact there than the FP32 bounds assume, and a
    // zero offset always takes the exact search
    constexpr double kVorMinOffset = 0x1p-28;
    constexpr int kVorNone = -99;  // no exit
    constexpr int kVorAsk = -98;   // not decided yet (Gen::resolve)

    // Tetrahedron record (indexed by cell, for the search of a position's cell and the start of a
    // path): vertices and outward face normals (TetraMeshSpatialGrid), density
    struct alignas(128) TetCell
    {
        double v[4][3];
        double dens;
        double pad[3];
        double n[4][3];
        double pad2[4];
    };
    static_assert(sizeof(TetCell) == 256, "tetra record must be 256 bytes");
    static_assert(offsetof(TetCell, n) == 128, "tetra normals start the second line");

    // One 64-byte record per face of a cell, at 4 * cell + face (the face opposite that vertex): its
    // normal, the cell behind it (-1: none), that cell's vertex opposite the face and density.  link:
    // bits 16-17 the face's number in that cell; bits 4e to 4e + 3, for a path that entered this cell
    // by face e, the place of the next cell's first and second vertex clockwise around the face in the
    // list (this cell's vertex e, then the two others of the face in this cell's clockwise order from
    // the one left out); bit 18 where the cells' vertices do not match and have to be read instead.
    struct alignas(64) TetFace
    {
        double n[3];
        int32_t cell;
        uint32_t link;
        double v[3];
        double dens;
    };
    static_assert(sizeof(TetFace) == 64, "tetra face record must be 64 bytes");


    // Consecutive "no exit found" steps after which a Voronoi or tetra path is ended.  The
    // reference steps by eps without limit; a path needs that many only when it has left the
    // valid geometry (such as a non-finite position).
    constexpr int kMaxNoExit = 4096;

    // One 64-byte record per octree node, indexed by node id.  A leaf holds everything a cell
    // crossing reads: its bounds, number density, cell index and, per wall, the node across it.  An
    // inner node holds its bounds, its first child and its split point (the upper corner of the first
    // child, TreeNode::leafChild's test point).  Bounds and split points are indices into the table
    // of the tree's distinct coordinates (GridView::planes: at most 3075 FP64 values for ten
    // levels, 1025 in a cube around the origin), which the kernels keep in LDS: a crossing reads half a cache line instead of a whole one, two
    // siblings share a line, and the 3.4e6 nodes of the spiral disk take 215 MB, less than the
    // last-level cache, instead of 430 MB.
    //
    // first[w] of a leaf: the neighbour itself where one leaf covers the wall; where several
    // smaller ones do, the node of the leaf's own size that they subdivide, so that a crossing
    // into a finer region descends by the split points (one record per level) instead of testing
    // the wall's list entry by entry; kOctNoNb at the domain boundary; kOctList where the table's
    // list is neither of these (the crossing then walks it).
    struct alignas(64) OctNode
    {
        int32_t lo[3], hi[3];  // bounds (planes)
        union
        {
            int32_t first[6];  // leaf: node across each wall (BACK..TOP)
            int32_t split[3];  // inner: split point (planes)
        };
        double dens;   // leaf: number density of the cell
        int32_t cell;  // leaf: cell index; inner: ~first child (children are 8 consecutive ids)
        int32_t pad;
    };
    static_assert(sizeof(OctNode) == 64, "node record must be half a cache line");
    static_assert(offsetof(OctNode, first) == 24 && offsetof(OctNode, dens) == 48 && offsetof(OctNode, cell) == 56,
                  "node record layout that OctRec reads");
    constexpr int32_t kOctNoNb = -1, kOctList = -2;
    constexpr int kLdsPlanes = 3200;  // coordinates kept in LDS at most (25.6 KB): ten levels have up to 3075

    // Read-only grid tables resident in HBM.  Octree: the node records and the leaves' neighbour
    // lists (node ids, sorted by decreasing overlap as TreeNode::sortNeighbors).
    struct GridView
    {
        double box[6];  // xmin, ymin, zmin, xmax, ymax, zmax of the domain
        double eps;     // 1e-12 * domain diagonal
        const double* xb;
        const double* yb;
        const double* zb;
        int nx, ny, nz;
        const double* dens;  // Cartesian: number density per cell
        const OctNode* node;
        const int32_t* leaf;  // cell -> node
        const double* planes;   // octree: the distinct coordinates of the tree's bounds; Cartesian: the
                                // borders of the three axes, one after the other
        int nplanes;
        int ldsPlanes;          // nonzero: the kernel staged them in LDS (stage_planes)
        const int32_t* nbOff;   // start of each node's and wall's neighbour list (6 per node, and the end)
        const int32_t* nbc;
        // Voronoi: cell records, neighbour entries and the block search lists (CSR over vbn^3
        // blocks of cell ids, in the reference's order)
        const VorCell* vcell;
        const VorNb* vnb;
        double vscale;  // 1 / the domain's largest side
        int vbn;
        const int32_t* vbl_off;
        const int32_t* vbl_id;
        // tetra: records and a block search grid (tbn^3 blocks, borders per axis, CSR of tetra
        // ids in increasing order)
        const TetCell* tcell;
        const TetFace* tface;
        int tbn;
        const double* tbx;
        const double* tby;
        const double* tbz;
        const int32_t* tbl_off;
        const int32_t* tbl_id;
    };

    // Box::cellIndices (Box.hpp:162-167) for the Voronoi block grid
    __device__ __forceinline__ int vor_block(const GridView& g, double x, double y, double z)
    {
        const int n = g.vbn;
        int i = static_cast<int>(n * (x - g.box[0]) / (g.box[3] - g.box[0]));
        int j = static_cast<int>(n * (y - g.box[1]) / (g.box[4] - g.box[1]));
        int k = static_cast<int>(n * (z - g.box[2]) / (g.box[5] - g.box[2]));
        i = max(0, min(n - 1, i));
        j = max(0, min(n - 1, j));
        k = max(0, min(n - 1, k));
        return i * n * n + j * n + k;
    }

    // the candidates' nearest site to a position, squared distance (r - site).norm2(), strict '<' (the
    // first of equal distances wins), four candidates in flight: its run, -1 if there is none
    __device__ __attribute__((noinline)) int vor_nearest(const VorCell* cell, const int32_t* ids, int q, int e, double x,
                                                         double y, double z)
    {
        int run = -1;
        double best = DBL_MAX;
        for (; q < e; q += 4)
        {
            int c[4];
            double d[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) c[u] = ids[min(q + u, e - 1)];
#pragma unroll
            for (int u = 0; u < 4; ++u)
            {
                const VorCell C = cell[c[u]];
                const double dx = x - C.x, dy = y - C.y, dz = z - C.z;
                d[u] = dx * dx + dy * dy + dz * dz;
                c[u] = C.run;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)  // (the last candidate again where fewer than four are left)
                if (d[u] < best)
                {
                    best = d[u];
                    run = c[u];
                }
        }
        return run;
    }

    // VoronoiMeshSnapshot::cellIndex: the run of the cell with the nearest site among the block's
    // candidates, -1 outside the domain
    __device__ __forceinline__ int vor_find(const GridView& g, double x, double y, double z)
    {
        if (!(x >= g.box[0] && x <= g.box[3] && y >= g.box[1] && y <= g.box[4] && z >= g.box[2] && z <= g.box[5]))
            return -1;
        const int b = vor_block(g, x, y, z);
        return vor_nearest(g.vcell, g.vbl_id, g.vbl_off[b], g.vbl_off[b + 1], x, y, z);
    }

    // number of borders <= v, minus one, clipped to a block index
    __device__ __forceinline__ int tet_axis_block(const double* bv, int n, double v)
    {
        int lo = 0, hi = n + 1;  // count of borders <= v lies in [lo, hi]
        while (lo < hi)
        {
            int mid = (lo + hi) >> 1;
            if (bv[mid] <= v)
                lo = mid + 1;
            else
                hi = mid;
        }
        return max(0, min(n - 1, lo - 1));
    }

    // Tetra::contains: bounding box of the vertices, then the face planes (outward normals;
    // faces 0..2 through vertex 3, face 3 through vertex 0)
    __device__ __forceinline__ bool tet_contains(const TetCell& T, double x, double y, double z)
    {
        double lx = DBL_MAX, ly = DBL_MAX, lz = DBL_MAX, hx = -DBL_MAX, hy = -DBL_MAX, hz = -DBL_MAX;
        for (int t = 0; t < 4; ++t)
        {
            lx = fmin(lx, T.v[t][0]);
            ly = fmin(ly, T.v[t][1]);
            lz = fmin(lz, T.v[t][2]);
            hx = fmax(hx, T.v[t][0]);
            hy = fmax(hy, T.v[t][1]);
            hz = fmax(hz, T.v[t][2]);
        }
        if (!(x >= lx && x <= hx && y >= ly && y <= hy && z >= lz && z <= hz)) return false;
        for (int f = 0; f <= 2; ++f)
            if ((T.v[3][0] - x) * T.n[f][0] + (T.v[3][1] - y) * T.n[f][1] + (T.v[3][2] - z) * T.n[f][2] < 0) return false;
        if ((T.v[0][0] - x) * T.n[3][0] + (T.v[0][1] - y) * T.n[3][1] + (T.v[0][2] - z) * T.n[3][2] < 0.) return false;
        return true;
    }

    // True when the point lies inside the tetra by a margin far above the rounding of the
    // face-plane tests: then no other tetra's tet_contains accepts it, so it is the one
    // tetra TetraMeshSpatialGrid::cellIndex returns.  The margin is 1e-13 of the summed
    // distances to the four vertices (a bound on the extent the rounding scales with).
    __device__ __forceinline__ bool tet_inside_strict(const TetCell& T, double x, double y, double z)
    {
        double scale = 0.;
        for (int t = 0; t < 4; ++t) scale += fabs(T.v[t][0] - x) + fabs(T.v[t][1] - y) + fabs(T.v[t][2] - z);
        const double tol = 1e-13 * scale;
        for (int f = 0; f <= 2; ++f)
            if (!((T.v[3][0] - x) * T.n[f][0] + (T.v[3][1] - y) * T.n[f][1] + (T.v[3][2] - z) * T.n[f][2] > tol)) return false;
        return (T.v[0][0] - x) * T.n[3][0] + (T.v[0][1] - y) * T.n[3][1] + (T.v[0][2] - z) * T.n[3][2] > tol;
    }

    // TetraMeshSpatialGrid::cellIndex: the lowest-index tetra containing the point (the
    // reference's search lists hold, in increasing index order, every tetra whose bounding
    // box meets the point's block, so its first hit is the lowest index; the block lists here
    // have the same property)
    __device__ __forceinline__ int tet_block(const GridView& g, double x, double y, double z)
    {
        const int n = g.tbn;
        return (tet_axis_block(g.tbx, n, x) * n + tet_axis_block(g.tby, n, y)) * n + tet_axis_block(g.tbz, n, z);
    }
    __device__ __forceinline__ int tet_cell_index(const GridView& g, double x, double y, double z)
    {
        const int b = tet_block(g, x, y, z);
        for (int q = g.tbl_off[b], e = g.tbl_off[b + 1]; q < e; ++q)
        {
            const int id = g.tbl_id[q];
            if (tet_contains(g.tcell[id], x, y, z)) return id;
        }
        return -1;
    }

    // TetraMeshSpatialGrid.cpp:44-50
    __host__ __device__ __forceinline__ void clockwise_vertices(int face, int& c0, int& c1, int& c2)
    {
        c0 = (face + 3) & 3;
        c1 = (face + 2) & 3;
        c2 = (face + 1) & 3;
        if ((face & 1) == 0)
        {
            int t = c0;
            c0 = c2;
            c2 = t;
        }
    }

    struct TetVert
    {
        double x, y, z;
        __device__ __forceinline__ void load(const double* v)
        {
            x = v[0];
            y = v[1];
            z = v[2];
        }
    };
    // a face record in registers
    struct TetFaceRec
    {
        double2 a, b, c, d;
        __device__ __forceinline__ void load(const TetFace* f)
        {
            const double2* p = reinterpret_cast<const double2*>(f);
            a = p[0];
            b = p[1];
            c = p[2];
            d = p[3];
        }
        __device__ __forceinline__ int cell() const { return __double2loint(b.y); }
        __device__ __forceinline__ uint32_t link() const { return static_cast<uint32_t>(__double2hiint(b.y)); }
    };

    enum GenState : int
    {
        kUnknown = 0,
        kInside = 1,
        kOutside = 2
    };

    // a ? x : b ? y : z on values (selecting among members by reference would make the
    // compiler select their addresses and keep the generator in scratch memory)
    template<typename T> __device__ __forceinline__ T pick3(bool a, bool b, T x, T y, T z)
    {
        const T yz = b ? y : z;
        return a ? x : yz;
    }
    __device__ __forceinline__ TetVert pick_vert(bool first, bool second, const TetVert& a, const TetVert& b, const TetVert& c)
    {
        return TetVert{pick3(first, second, a.x, b.x, c.x), pick3(first, second, a.y, b.y, c.y),
                       pick3(first, second, a.z, b.z, c.z)};
    }

    // a / b for a correctly rounded reciprocal y = RN(1 / b): the product with y, one Newton step
    // that makes the quotient faithful, and Markstein's correction with the exact remainder, which
    // gives the correctly rounded quotient -- the same value as the division (P. Markstein, IBM
    // J. Res. Dev. 34, 1990), in five FP64 operations instead of the division's eleven.  Positions
    // and directions along a path share the three divisors, so y is made once per path.
    __device__ __forceinline__ double quotient(double a, double b, double y)
    {
        double q = a * y;
        q = fma(fma(-b, q, a), y, q);
        return fma(fma(-b, q, a), y, q);
    }

    // The coordinate table of a Cartesian grid or octree in LDS (dynamic shared memory of nplanes
    // doubles when GridView::ldsPlanes is set); every kernel that walks a grid calls stage_planes
    // first.
    extern __shared__ double skg_planes[];

    template<int GT> __device__ __forceinline__ void stage_planes(const GridView& g)
    {
        if constexpr (GT == kOctree || GT == kCartesian)
        {
            if (g.ldsPlanes)
                for (int t = threadIdx.x; t < g.nplanes; t += blockDim.x) skg_planes[t] = g.planes[t];
            __syncthreads();
        }
    }

    // What a crossing reads of an octree node's record, in registers (no member is selected by
    // reference, which would leave the record in scratch memory)
    struct OctRec
    {
        int4 a, b, c, d;
        __device__ __forceinline__ void load(const OctNode* nd)
        {
            const int4* p = reinterpret_cast<const int4*>(nd);
            a = p[0];
            b = p[1];
            c = p[2];
            d = p[3];
        }
        __device__ __forceinline__ int cell() const { return d.z; }
        __device__ __forceinline__ double dens() const { return __hiloint2double(d.y, d.x); }
    };

    // bounds of a node
    struct OctBox
    {
        double x0, y0, z0, x1, y1, z1;
        __device__ __forceinline__ void load(const GridView& g, const OctRec& R)
        {
            if (g.ldsPlanes)
            {
                x0 = skg_planes[R.a.x];
                y0 = skg_planes[R.a.y];
                z0 = skg_planes[R.a.z];
                x1 = skg_planes[R.a.w];
                y1 = skg_planes[R.b.x];
                z1 = skg_planes[R.b.y];
            }
            else
            {
                x0 = g.planes[R.a.x];
                y0 = g.planes[R.a.y];
                z0 = g.planes[R.a.z];
                x1 = g.planes[R.a.w];
                y1 = g.planes[R.b.x];
                z1 = g.planes[R.b.y];
            }
        }
        __device__ __forceinline__ bool closed_contains(double x, double y, double z) const
        {
            return x >= x0 && x <= x1 && y >= y0 && y <= y1 && z >= z0 && z <= z1;
        }
    };

    // TreeNode::leafChild from the root (TreeSpatialGrid.cpp:190-219, OctTreeNode.cpp:37-42): the
    // leaf containing the position by the half-open rule of the split points, -1 outside the
    // root's closed box
    __device__ __forceinline__ int oct_search(const OctNode* node, const double* planes, double x, double y, double z)
    {
        if (!(x >= planes[node->lo[0]] && x <= planes[node->hi[0]] && y >= planes[node->lo[1]]
              && y <= planes[node->hi[1]] && z >= planes[node->lo[2]] && z <= planes[node->hi[2]]))
            return -1;
        int nd = 0;
        while (true)
        {
            const OctNode& N = node[nd];
            const int c = N.cell;
            if (c >= 0) return nd;
            nd = ~c + (x < planes[N.split[0]] ? 0 : 1) + (y < planes[N.split[1]] ? 0 : 2)
                 + (z < planes[N.split[2]] ? 0 : 4);
        }
    }

    struct OctNext
    {
        int node;
        double x, y, z;
    };

    // The next leaf after a crossing of wall `wall` of leaf i at the position (x, y, z), by the
    // reference's own sequence (TreeSpatialGrid.cpp:184-219): the wall's neighbour list in order,
    // then the search from the root, then, still in leaf i, the same search with the position one
    // ulp further along the path; node -1 where the path ends.  Called where the crossing's shorter
    // rules do not decide (a position on a split plane or outside the node across the wall), and
    // kept out of the crossing's registers.
    __device__ __attribute__((noinline)) OctNext oct_next_exact(const OctNode* node, const double* planes,
                                                                const int32_t* nbOff, const int32_t* nbc, int i, int wall,
                                                                double x, double y, double z, double kx, double ky,
                                                                double kz)
    {
        int c = -2;
        const int64_t at = 6 * static_cast<int64_t>(i) + wall;
        for (int q = nbOff[at], e = nbOff[at + 1]; q < e; ++q)
        {
            const int id = nbc[q];
            const OctNode& N = node[id];
            if (x >= planes[N.lo[0]] && x <= planes[N.hi[0]] && y >= planes[N.lo[1]] && y <= planes[N.hi[1]]
                && z >= planes[N.lo[2]] && z <= planes[N.hi[2]])
            {
                c = id;
                break;
            }
        }
        if (c == -2) c = oct_search(node, planes, x, y, z);
        if (c == i)
        {
            x = nextafter(x, (kx < 0.) ? -DBL_MAX : DBL_MAX);
            y = nextafter(y, (ky < 0.) ? -DBL_MAX : DBL_MAX);
            z = nextafter(z, (kz < 0.) ? -DBL_MAX : DBL_MAX);
            c = oct_search(node, planes, x, y, z);
        }
        return OctNext{c == i ? -1 : c, x, y, z};
    }

    struct VorExit
    {
        int id;
        double s;
    };

    // Exit distance through the bisector plane between the sites p and e (0 where the plane is
    // not ahead), or through domain wall id (VoronoiMeshSnapshot.cpp:1119-1170)
    __device__ __forceinline__ double vor_bisector(double px, double py, double pz, double ex, double ey, double ez,
                                                   double rx, double ry, double rz, double kx, double ky, double kz)
    {
        const double nx = ex - px, ny = ey - py, nz = ez - pz;
        const double ndotk = nx * kx + ny * ky + nz * kz;
        if (!(ndotk > 0)) return 0.;
        const double qx = 0.5 * (ex + px), qy = 0.5 * (ey + py), qz = 0.5 * (ez + pz);
        return (nx * (qx - rx) + ny * (qy - ry) + nz * (qz - rz)) / ndotk;
    }
    __device__ __forceinline__ double vor_wall(const double* box, int id, double rx, double ry, double rz, double kx,
                                               double ky, double kz)
    {
        const int w = -1 - id;  // 0..5: xmin, xmax, ymin, ymax, zmin, zmax
        if (w >= 6) return 0.;
        // (selected as values: a selection among the members' addresses made the pipeline's trace kernel
        // keep its whole parameter block in scratch memory, 912 bytes per lane)
        const bool up = w & 1;
        const double x0 = box[0], y0 = box[1], z0 = box[2], x1 = box[3], y1 = box[4], z1 = box[5];
        const double face = pick3(w < 2, w < 4, up ? x1 : x0, up ? y1 : y0, up ? z1 : z0);
        const double r = pick3(w < 2, w < 4, rx, ry, rz), k = pick3(w < 2, w < 4, kx, ky, kz);
        return (face - r) / k;
    }

    // The exit of the cell with the run at slot i from the exact distances of all its neighbours:
    // the smallest positive one, the first of equal ones (kVorNone if none is positive).  Called
    // where the FP32 bounds leave more than one neighbour, and kept out of the crossing's registers.
    __device__ __attribute__((noinline)) int vor_exit_exact(const VorNb* nb, double b0, double b1, double b2, double b3,
                                                            double b4, double b5, int i, double rx, double ry, double rz,
                                                            double kx, double ky, double kz)
    {
        const double box[6] = {b0, b1, b2, b3, b4, b5};
        const VorHead& C = *reinterpret_cast<const VorHead*>(nb + i);
        int out = kVorNone;
        double best = DBL_MAX;
        for (int q = i + 3; q < i + 3 + C.count; ++q)
        {
            const int id = nb[q].id;
            double s;
            if (id >= 0)
            {
                const VorHead& N = *reinterpret_cast<const VorHead*>(nb + id);
                s = vor_bisector(C.x, C.y, C.z, N.x, N.y, N.z, rx, ry, rz, kx, ky, kz);
            }
            else
                s = vor_wall(box, id, rx, ry, rz, kx, ky, kz);
            if (s > 0 && s < best)
            {
                best = s;
                out = id;
            }
        }
        return out;
    }

    // the value of the first of each group of L lanes (1 or 4), in every lane of the group
    template<int L> __device__ __forceinline__ int group_first(int v)
    {
        if constexpr (L == 1) return v;
        return __builtin_amdgcn_update_dpp(v, v, 0x00, 0xF, 0xF, true);  // quad_perm 0 0 0 0
    }
    template<int L> __device__ __forceinline__ double group_first(double v)
    {
        return __hiloint2double(group_first<L>(__double2hiint(v)), group_first<L>(__double2loint(v)));
    }

    // a cell's run: the head, and the lane's entries of the first L * kVorAhead<L>
    template<int L> struct VorRun
    {
        double2 a, b;
        float4 c;
        float4 f[kVorAhead<L>];
        __device__ __forceinline__ void load_entries(const VorNb* p)
        {
#pragma unroll
            for (int u = 0; u < kVorAhead<L>; ++u) f[u] = *reinterpret_cast<const float4*>(p + u * L);
        }
        __device__ __forceinline__ void load(const GridView& g, int slot, int sub)
        {
            const VorNb* p = g.vnb + slot;
            a = *reinterpret_cast<const double2*>(p);
            b = *reinterpret_cast<const double2*>(p + 1);
            c = *reinterpret_cast<const float4*>(p + 2);
            load_entries(p + 3 + sub);
        }
        __device__ __forceinline__ int count() const { return __float_as_int(c.x); }
        __device__ __forceinline__ int cell() const { return __float_as_int(c.y); }
    };

    // The exit search in FP32 (lengths in units of the domain's side).  With the offset n of a
    // neighbour's site and w of the position from the cell's site, the bisector is at the distance
    // a = n.(n / 2 - w) / n.k.  The numerator is off by at most En = eps (r2 + w.w) and the
    // denominator by Ed = eps r1 |k|, with the cell's largest n.n (r2) and 1-norm (r1); where the
    // denominator exceeds 6 Ed, a is then off by at most 2 (En + a Ed) / n.k.  A denominator below
    // -4 Ed makes the neighbour no exit.  One between the two (a face parallel to the path) makes it an
    // exit at any distance from (num - En) / 7 Ed on, which the same formula with 6 Ed as the
    // denominator stays below, or no exit at all.  (Without that bound, which the walls' cells of every
    // mesh need, such crossings went to the exact search.  2^18 packets seen face-on and at 60 degrees,
    // lattice of 36^3 sites: 26.6 -> 11.4 ms; and edge-on, 60 000 sites: 32.5 -> 23.6 ms.)
    struct VorSearch
    {
        float wx, wy, wz, fx, fy, fz, en2, ed2, ed4, ed6;
        float l1, l2, a1, mn;  // the two smallest lower bounds, the first one's distance; the smallest numerator
        int id;

        // valid: the entry is one (false: read past the end of the run)
        __device__ __forceinline__ void entry(const float4& v, bool valid)
        {
            const float num = fmaf(v.x, fmaf(0.5f, v.x, -wx), fmaf(v.y, fmaf(0.5f, v.y, -wy), v.z * fmaf(0.5f, v.z, -wz)));
            const float den = fmaf(v.x, fx, fmaf(v.y, fy, v.z * fz));
            const float r = __builtin_amdgcn_rcpf(fmaxf(den, ed6));
            float a = num * r;
            float lb = fmaf(-r, fmaf(a, ed2, en2), a);
            lb = valid && den >= -ed4 ? lb : INFINITY;
            a = den > ed6 ? a : INFINITY;  // no upper bound
            const bool first = lb < l1;
            l2 = __builtin_amdgcn_fmed3f(l1, lb, l2);
            l1 = first ? lb : l1;
            a1 = first ? a : a1;
            id = first ? __float_as_int(v.w) : id;
            mn = fminf(mn, valid ? num : INFINITY);
        }

        // with the search of the lane that quad_perm CTRL names
        template<int CTRL> __device__ __forceinline__ void merge()
        {
            const float ol1 = other<CTRL>(l1), ol2 = other<CTRL>(l2), oa1 = other<CTRL>(a1);
            const int oid = __builtin_amdgcn_update_dpp(id, id, CTRL, 0xF, 0xF, true);
            mn = fminf(mn, other<CTRL>(mn));
            l2 = fminf(fminf(l2, ol2), fmaxf(l1, ol1));
            const bool first = ol1 < l1;
            l1 = first ? ol1 : l1;
            a1 = first ? oa1 : a1;
            id = first ? oid : id;
        }
        template<int CTRL> static __device__ __forceinline__ float other(float v)
        {
            const int w = __float_as_int(v);
            return __int_as_float(__builtin_amdgcn_update_dpp(w, w, CTRL, 0xF, 0xF, true));
        }
    };

    // L: the lanes that walk a path together, all with the same state (Voronoi: each searches a share
    // of the neighbours)
    template<int GT, int L = 1> struct Gen
    {
        double rx, ry, rz, kx, ky, kz;
        int state;
        int i, j, k;  // Cartesian: entry of the border ahead on each axis in the planes table; octree: i = current leaf's node; Voronoi: i = the
                      // current cell's run, j = the run or wall behind its exit, k = the
                      // steps without exit; tetra: i = current
                      // cell, j = entering face, -1 at the end, k = the steps without exit
        double sx, sy, sz;      // Voronoi: the current cell's site
        double ikx, iky, ikz;   // Cartesian, octree: reciprocals of the direction
        double b0, b1, b2;      // Cartesian, octree: the current cell's wall ahead on each axis
        double bn;              // the current cell's density
        TetVert V, C0, C1, C2;  // tetra: the vertex opposite the entering face, that face's clockwise
        bool ask;               // tetra: something to resolve()
        int f0, f1, f2;         // octree: the node across each of those walls
        int cell;               // Cartesian, octree, Voronoi: the current cell's index
        uint32_t pend;  // octree: a node to descend into next and the crossed wall (node << 3 | wall),
                        // or kNoPend
        int hint;  // a cell that probably contains the start point (-1: none), after the first step
                   // the start cell: octree a node, Voronoi a run (a hint that resolve() had to replace
                   // stays: the position is then so near a face that its own cell would be rejected too),
                   // tetra a cell, Cartesian the cell's indices i | j << 10 | k << 20 (no more than 1024
                   // cells along an axis)
        static constexpr uint32_t kNoPend = 0xFFFFFFFFu;  // node ids stay below 2^29

        __device__ __forceinline__ void start(double r0, double r1, double r2, double k0, double k1, double k2,
                                              int start_hint = -1)
        {
            hint = start_hint;
            rx = r0;
            ry = r1;
            rz = r2;
            kx = k0;
            ky = k1;
            kz = k2;
            state = kUnknown;
        }

        __device__ __forceinline__ bool move_inside(const GridView& g, double& cumds)
        {
            const double eps = g.eps;
            state = kOutside;
            cumds = 0.;
            if (rx <= g.box[0])
            {
                if (kx <= 0.0) return false;
                double d = (g.box[0] - rx) / kx;
                rx = g.box[0] + eps;
                ry += ky * d;
                rz += kz * d;
                cumds += d;
            }
            else if (rx >= g.box[3])
            {
                if (kx >= 0.0) return false;
                double d = (g.box[3] - rx) / kx;
                rx = g.box[3] - eps;
                ry += ky * d;
                rz += kz * d;
                cumds += d;
            }
            if (ry <= g.box[1])
            {
                if (ky <= 0.0) return false;
                double d = (g.box[1] - ry) / ky;
                rx += kx * d;
                ry = g.box[1] + eps;
                rz += kz * d;
                cumds += d;
            }
            else if (ry >= g.box[4])
            {
                if (ky >= 0.0) return false;
                double d = (g.box[4] - ry) / ky;
                rx += kx * d;
                ry = g.box[4] - eps;
                rz += kz * d;
                cumds += d;
            }
            if (rz <= g.box[2])
            {
                if (kz <= 0.0) return false;
                double d = (g.box[2] - rz) / kz;
                rx += kx * d;
                ry += ky * d;
                rz = g.box[2] + eps;
                cumds += d;
            }
            else if (rz >= g.box[5])
            {
                if (kz >= 0.0) return false;
                double d = (g.box[5] - rz) / kz;
                rx += kx * d;
                ry += ky * d;
                rz = g.box[5] - eps;
                cumds += d;
            }
            if (!(rx >= g.box[0] && rx <= g.box[3] && ry >= g.box[1] && ry <= g.box[4] && rz >= g.box[2]
                  && rz <= g.box[5]))
                return false;
            state = kInside;
            return true;
        }

        // ---------------------------------------------------------------- octree
        // the leaf nd becomes the current one: of its record, the crossing needs only the wall
        // ahead on each axis (the direction does not change along a path) -- its coordinate
        // (TreeSpatialGrid.cpp:157-159) and the node across it -- the density and the cell
        __device__ __forceinline__ void adopt(const OctRec& R, const OctBox& B, int nd)
        {
            i = nd;
            cell = R.cell();
            b0 = (kx < 0.0) ? B.x0 : B.x1;
            b1 = (ky < 0.0) ? B.y0 : B.y1;
            b2 = (kz < 0.0) ? B.z0 : B.z1;
            bn = R.dens();
            f0 = (kx < 0.0) ? R.b.z : R.b.w;
            f1 = (ky < 0.0) ? R.c.x : R.c.y;
            f2 = (kz < 0.0) ? R.c.z : R.c.w;
            pend = kNoPend;
        }

        // the start leaf: the hint, when the point lies in its box the way the top-down search
        // assigns points to leaves -- lo <= r < hi on each axis (a point on a split plane goes to
        // the upper child), hi included at the domain's upper boundary, so that every split plane
        // of the leaf's ancestors sends the search toward it -- else the search's leaf
        __device__ __forceinline__ bool oct_begin(const GridView& g)
        {
            OctRec R;
            OctBox B;
            int nd = hint;
            bool found = false;
            if (nd >= 0)
            {
                R.load(g.node + nd);
                B.load(g, R);
                const bool inx = rx >= B.x0 && (rx < B.x1 || B.x1 == g.box[3]);
                const bool iny = ry >= B.y0 && (ry < B.y1 || B.y1 == g.box[4]);
                const bool inz = rz >= B.z0 && (rz < B.z1 || B.z1 == g.box[5]);
                found = inx && iny && inz;
            }
            if (!found)
            {
                nd = oct_search(g.node, g.planes, rx, ry, rz);
                if (nd < 0) return false;
                R.load(g.node + nd);
                B.load(g, R);
            }
            adopt(R, B, nd);
            hint = nd;
            return true;
        }

        // One step of the octree generator (TreeSpatialGrid::MySegmentGenerator::next,
        // TreeSpatialGrid.cpp:143-228), with one dependent record load: the crossing of the current
        // leaf and the record of the node across the exit wall, or one level of the descent into a
        // finer region.  Returns as cross() does.
        __device__ __forceinline__ int cross_octree(const GridView& g, int& m, double& ds, double& n)
        {
            int out = 0;
            int nd = static_cast<int>(pend >> 3), wall = static_cast<int>(pend & 7u);
            if (pend == kNoPend)
            {
                // exit distance along each axis to the wall ahead, (wall - r) / k, or DBL_MAX for a
                // component within 1e-15 of zero; the smallest wins with the ties of
                // TreeSpatialGrid.cpp:157-181
                const double dsx = fabs(kx) > 1e-15 ? quotient(b0 - rx, kx, ikx) : DBL_MAX;
                const double dsy = fabs(ky) > 1e-15 ? quotient(b1 - ry, ky, iky) : DBL_MAX;
                const double dsz = fabs(kz) > 1e-15 ? quotient(b2 - rz, kz, ikz) : DBL_MAX;
                const bool ax = dsx <= dsy && dsx <= dsz;
                const bool ay = !ax && dsy <= dsx && dsy <= dsz;
                const double d = pick3(ax, ay, dsx, dsy, dsz);
                wall = pick3(ax, ay, (kx < 0.0) ? 0 : 1, (ky < 0.0) ? 2 : 3, (kz < 0.0) ? 4 : 5);
                nd = pick3(ax, ay, f0, f1, f2);
                const double step = d + g.eps;
                rx += kx * step;
                ry += ky * step;
                rz += kz * step;
                m = cell;
                ds = d;
                n = bn;
                out = 1;
                // a wall without neighbours is on the domain's boundary: outside the root's closed
                // box the search finds no leaf (TreeNode::leafChild), and the path ends here
                if (nd == kOctNoNb
                    && !(rx >= g.box[0] && rx <= g.box[3] && ry >= g.box[1] && ry <= g.box[4] && rz >= g.box[2]
                         && rz <= g.box[5]))
                {
                    state = kOutside;
                    return 2;
                }
            }
            OctRec R;
            OctBox B;
            R.load(g.node + max(nd, 0));
            B.load(g, R);
            const bool closed = nd >= 0 && B.closed_contains(rx, ry, rz);
            const int c = R.cell();
            if (__builtin_expect(closed && c >= 0, 1))
            {
                // the neighbour contains the new position (TreeNode::neighbor, TreeNode.cpp:103-112)
                adopt(R, B, nd);
                return out;
            }
            if (closed)
            {
                // off the split planes exactly one of the finer neighbours contains the position
                const double sx = g.planes[R.b.z], sy = g.planes[R.b.w], sz = g.planes[R.c.x];
                if (__builtin_expect(rx != sx && ry != sy && rz != sz, 1))
                {
                    pend = static_cast<uint32_t>(~c + (rx < sx ? 0 : 1) + (ry < sy ? 0 : 2) + (rz < sz ? 0 : 4)) << 3
                           | static_cast<uint32_t>(wall);
                    return out;
                }
            }
            const OctNext e = oct_next_exact(g.node, g.planes, g.nbOff, g.nbc, i, wall, rx, ry, rz, kx, ky, kz);
            nd = e.node;
            rx = e.x;
            ry = e.y;
            rz = e.z;
            if (nd < 0)
            {
                state = kOutside;
                return out ? 2 : -1;
            }
            R.load(g.node + nd);
            B.load(g, R);
            adopt(R, B, nd);
            return out;
        }

        // ---------------------------------------------------------------- all grids
        // Enters the domain and finds the start cell; false when the path has no segment at all.
        // entry: the length of the path before the domain (0 when it starts inside).
        __device__ __forceinline__ bool begin(const GridView& g, double& entry)
        {
            if (!move_inside(g, entry)) return false;
            if constexpr (GT == kCartesian || GT == kOctree)
            {
                ikx = 1. / kx;
                iky = 1. / ky;
                ikz = 1. / kz;
            }
            if constexpr (GT == kCartesian)
            {
                const int oy = g.nx + 1, oz = oy + g.ny + 1;
                int ci = hint & 1023, cj = (hint >> 10) & 1023, ck = hint >> 20;
                const bool found = hint >= 0 && rx >= border(g, ci) && rx < border(g, ci + 1) && ry >= border(g, oy + cj)
                                   && ry < border(g, oy + cj + 1) && rz >= border(g, oz + ck) && rz < border(g, oz + ck + 1);
                if (!found)
                {
                    ci = locate(g, 0, g.nx, rx);
                    cj = locate(g, oy, g.ny, ry);
                    ck = locate(g, oz, g.nz, rz);
                }
                hint = max(max(g.nx, g.ny), g.nz) <= 1024 ? ci | (cj << 10) | (ck << 20) : -1;
                cell = ck + g.nz * cj + g.nz * g.ny * ci;
                i = ci + (kx < 0.0 ? 0 : 1);
                j = g.nx + 1 + cj + (ky < 0.0 ? 0 : 1);
                k = g.nx + g.ny + 2 + ck + (kz < 0.0 ? 0 : 1);
                b0 = border(g, i);
                b1 = border(g, j);
                b2 = border(g, k);
                bn = g.dens ? g.dens[cell] : 0.;
            }
            else if constexpr (GT == kOctree)
            {
                if (!oct_begin(g))
                {
                    state = kOutside;
                    return false;
                }
            }
            else
            {
                if constexpr (GT == kVoronoi)
                {
                    // the first step enters the cell, and finds out whether the hint is right
                    i = hint >= 0 ? kVorHinted : kVorEnter;
                    if (hint < 0) hint = vor_find(g, rx, ry, rz);
                    j = hint;
                    k = 0;
                }
                else
                {
                    i = hint >= 0 && tet_inside_strict(g.tcell[hint], rx, ry, rz) ? hint : tet_cell_index(g, rx, ry, rz);
                    hint = i;
                    k = 0;
                    ask = false;
                    if (i >= 0) tet_enter(g, -1);
                }
                if (hint < 0)
                {
                    state = kOutside;
                    return false;
                }
            }
            return true;
        }

        // One step of a path that has begun: 1 with the segment (the cell m, the length ds and the
        // cell's number density n) when the step completed one, 2 with the path's last segment, 0
        // when it only progressed (the octree's descent), -1 at the end of the path.
        __device__ __forceinline__ int cross(const GridView& g, int& m, double& ds, double& n)
        {
            if constexpr (GT == kOctree)
                return cross_octree(g, m, ds, n);
            else if constexpr (GT == kVoronoi)
                return cross_voronoi(g, m, ds, n);
            else if constexpr (GT == kTetra)
                return cross_tetra(g, m, ds, n);
            else
                return !next_cartesian(g, m, ds, n) ? -1 : state == kOutside ? 2 : 1;
        }

        // One step of a path from its start on, as cross(); the first step begins the path and
        // returns its segment before the domain, if any (m = -1).
        __device__ __forceinline__ int advance(const GridView& g, int& m, double& ds, double& n)
        {
            if (state == kInside && asks()) resolve(g);
            return step(g, m, ds, n);
        }
        // likewise, where the caller looks after asks()
        __device__ __forceinline__ int step(const GridView& g, int& m, double& ds, double& n)
        {
            if (state == kOutside) return -1;
            if (state == kUnknown)
            {
                double entry;
                if (!begin(g, entry)) return -1;
                if (entry > 0.)
                {
                    m = -1;
                    ds = entry;
                    n = 0.;
                    return 1;
                }
            }
            return cross(g, m, ds, n);
        }

        __device__ __forceinline__ static double border(const GridView& g, int q)
        {
            return g.ldsPlanes ? skg_planes[q] : g.planes[q];
        }

        // NR::locateClip (NR.hpp:130-144, :177-183) over the n + 1 borders from entry `first` on: the
        // cell that holds x
        __device__ __forceinline__ static int locate(const GridView& g, int first, int n, double x)
        {
            if (x < border(g, first)) return 0;
            int jl = -1, ju = n;
            while (ju - jl > 1)
            {
                const int jm = (ju + jl) >> 1;
                if (x < border(g, first + jm))
                    ju = jm;
                else
                    jl = jm;
            }
            return jl;
        }

        // CartesianSpatialGrid.cpp:77-153.  The border ahead on each axis and the cell's density are
        // kept from crossing to crossing: a crossing reads one border (of the axis it moved along,
        // from LDS) and the next cell's density, which is needed only when that cell's segment is
        // complete, so that its load is in flight during the next crossing's arithmetic.
        __device__ __forceinline__ bool next_cartesian(const GridView& g, int& m, double& ds, double& n)
        {
            const double dsx = (fabs(kx) > 1e-15) ? quotient(b0 - rx, kx, ikx) : DBL_MAX;
            const double dsy = (fabs(ky) > 1e-15) ? quotient(b1 - ry, ky, iky) : DBL_MAX;
            const double dsz = (fabs(kz) > 1e-15) ? quotient(b2 - rz, kz, ikz) : DBL_MAX;
            m = cell;
            n = bn;
            const bool ax = dsx <= dsy && dsx <= dsz;
            const bool ay = !ax && dsy < dsx && dsy <= dsz;
            ds = pick3(ax, ay, dsx, dsy, dsz);
            rx = ax ? b0 : rx + kx * ds;
            ry = ay ? b1 : ry + ky * ds;
            rz = (ax || ay) ? rz + kz * ds : b2;
            const bool neg = pick3(ax, ay, kx, ky, kz) < 0.0;
            const int first = pick3(ax, ay, 0, g.nx + 1, g.nx + g.ny + 2), count = pick3(ax, ay, g.nx, g.ny, g.nz);
            const int at = pick3(ax, ay, i, j, k);
            if (at == (neg ? first : first + count))
            {
                state = kOutside;  // the domain's border
                return true;
            }
            const int to = at + (neg ? -1 : 1);
            const int stride = pick3(ax, ay, g.nz * g.ny, g.nz, 1);
            cell += neg ? -stride : stride;
            bn = g.dens ? g.dens[cell] : 0.;
            const double b = border(g, to);
            i = ax ? to : i;
            j = ay ? to : j;
            k = (ax || ay) ? k : to;
            b0 = ax ? b : b0;
            b1 = ay ? b : b1;
            b2 = (ax || ay) ? b2 : b;
            return true;
        }

        // One step of the Voronoi generator (VoronoiMeshSnapshot.cpp:1119-1210): the crossing of the
        // current cell through its exit, found by the step before, and the search of the exit of the
        // cell behind it; the first step only does the latter.  Returns as cross() does.
        //
        // Bound by the vector memory path: the runs of the lanes lie apart, so each 16-byte load
        // returns at about one lane a cycle (the return path was busy 80 % of the time with FP64
        // sites), then by the latency of the run's lines, as the table does not fit the L2.  Hence
        // 16-byte entries and one dependent read per step: the entries name their neighbours' runs,
        // not their cells, and the exact exit distance takes the neighbour's site from the run that
        // is read anyway.  400 000 sites, 2^18 packets, tau 5: 90 -> 40 ms; 2000 optical
        // depths through 60 000 sites with four lanes each: 0.47 -> 0.25 ms.
        static constexpr int kVorHinted = -1, kVorEnter = -2;  // i before the first step
        __device__ __forceinline__ int cross_voronoi(const GridView& g, int& m, double& ds, double& n)
        {
            if (__builtin_expect(j == kVorNone, 0))
            {
                state = kOutside;
                return -1;
            }
            const int sub = L > 1 ? static_cast<int>(threadIdx.x) & (L - 1) : 0;
            VorRun<L> R;
            R.load(g, max(j, 0), sub);
            const bool hinted = i == kVorHinted;
            int out = 0;
            if (i >= 0)
            {
                const double d = j >= 0 ? vor_bisector(sx, sy, sz, R.a.x, R.a.y, R.b.x, rx, ry, rz, kx, ky, kz)
                                        : vor_wall(g.box, j, rx, ry, rz, kx, ky, kz);
                const double step = d + g.eps;
                rx += kx * step;
                ry += ky * step;
                rz += kz * step;
                m = cell;
                ds = d;
                n = bn;
                out = 1;
                k = 0;
                if (j < 0)
                {
                    state = kOutside;
                    return 2;
                }
            }
            const int run = j;
            if (!hinted) i = run;
            sx = R.a.x;
            sy = R.a.y;
            sz = R.b.x;
            bn = R.b.y;
            cell = R.cell();
            VorSearch S;
            S.wx = static_cast<float>((rx - sx) * g.vscale);
            S.wy = static_cast<float>((ry - sy) * g.vscale);
            S.wz = static_cast<float>((rz - sz) * g.vscale);
            S.fx = static_cast<float>(kx);
            S.fy = static_cast<float>(ky);
            S.fz = static_cast<float>(kz);
            const float kk = fabsf(S.fx) + fabsf(S.fy) + fabsf(S.fz);
            S.en2 = 2.f * kVorEps * fmaf(S.wx, S.wx, fmaf(S.wy, S.wy, fmaf(S.wz, S.wz, R.c.z)));
            S.ed2 = 2.f * kVorEps * kk * R.c.w;
            S.ed4 = 2.f * S.ed2;
            S.ed6 = 3.f * S.ed2;
            S.l1 = S.l2 = S.mn = INFINITY;
            S.a1 = 0.f;
            S.id = kVorNone;
#pragma unroll
            for (int u = 0; u < kVorAhead<L>; ++u) S.entry(R.f[u], (u + 1) * L <= kVorPad || u * L + sub < R.count());
            for (int q = L * kVorAhead<L>; q < R.count(); q += L * kVorAhead<L>)
            {
                R.load_entries(g.vnb + run + 3 + q + sub);
#pragma unroll
                for (int u = 0; u < kVorAhead<L>; ++u) S.entry(R.f[u], q + u * L + sub < R.count());
            }
            if constexpr (L == 4)
            {
                S.template merge<0xB1>();  // quad_perm 1 0 3 2
                S.template merge<0x4E>();  // quad_perm 2 3 0 1
            }
            // the hint holds where the position is clearly nearer to the site than to every
            // neighbour's (half the difference of the squared distances is the numerator): inside
            // the domain, the cell is the set of points nearer to its site than to the sites
            // across its faces, so that site is then the nearest of all
            const bool there = !hinted || S.mn > S.en2;
            // one neighbour is nearer than all the others can be (none at all: resolve() steps on)
            const bool one = S.id != kVorNone && S.l1 > 0.f && 1.00001f * (2.f * S.a1 - S.l1) < S.l2 && kk > 1e-12f && kk < 1e12f;
            j = kVorAsk;
            if (there)
            {
                i = run;
                if (one) j = S.id;
            }
            return out;
        }

        // Whether the step left something to resolve() before the next step: an exit, or a start cell,
        // that the Voronoi search could not decide in FP32; a tetra position without an exit, or vertices to read.  Apart
        // from the step, so that no call and no cell search lies in the loop of the crossings (the
        // registers saved around a call were half of the Voronoi loop's time).
        __device__ __forceinline__ bool asks() const
        {
            return GT == kVoronoi ? j == kVorAsk : GT == kTetra ? ask : false;
        }
        // no path: nothing to resolve
        __device__ __forceinline__ void idle()
        {
            if constexpr (GT == kVoronoi) j = kVorNone;
            if constexpr (GT == kTetra) ask = false;
        }
        __device__ __forceinline__ void resolve(const GridView& g)
        {
            if constexpr (GT == kVoronoi)
            {
                if (i >= 0)
                {
                    j = vor_exit_exact(g.vnb, g.box[0], g.box[1], g.box[2], g.box[3], g.box[4], g.box[5], i, rx, ry, rz,
                                       kx, ky, kz);
                    if (j != kVorNone) return;
                    if (!nudge(g)) return;
                }
                i = kVorEnter;
                j = vor_find(g, rx, ry, rz);
                if (j < 0) j = kVorNone;
            }
            else if constexpr (GT == kTetra)
            {
                ask = false;
                if (k == kTetReload)
                {
                    k = 0;
                    tet_enter(g, j);
                    return;
                }
                j = -1;
                if (!nudge(g)) return;
                i = tet_cell_index(g, rx, ry, rz);
                if (i >= 0) tet_enter(g, -1);
            }
        }
        // a step of eps along the path; false after too many without an exit
        __device__ __forceinline__ bool nudge(const GridView& g)
        {
            rx += kx * g.eps;
            ry += ky * g.eps;
            rz += kz * g.eps;
            return ++k < kMaxNoExit;
        }

        // Tetra::findEnteringFace: the first of the six edges with a nonzero Pluecker product
        __device__ __forceinline__ int entering_face(const TetCell& T) const
        {
            int e = 0;
            for (int t1 = 0; t1 < 3; t1++)
                for (int t2 = t1 + 1; t2 < 4; t2++)
                {
                    double wx = rx - T.v[t1][0], wy = ry - T.v[t1][1], wz = rz - T.v[t1][2];
                    double mx = ky * wz - kz * wy, my = kz * wx - kx * wz, mz = kx * wy - ky * wx;
                    double prod = mx * (T.v[t2][0] - T.v[t1][0]) + my * (T.v[t2][1] - T.v[t1][1])
                                  + mz * (T.v[t2][2] - T.v[t1][2]);
                    if (prod != 0.)
                    {
                        // etable {{3,2},{1,3},{2,1},{3,0},{0,2},{1,0}} (TetraMeshSpatialGrid.cpp:91)
                        constexpr int neg = 3 | (1 << 2) | (2 << 4) | (3 << 6) | (0 << 8) | (1 << 10);
                        constexpr int pos = 2 | (3 << 2) | (1 << 4) | (0 << 6) | (2 << 8) | (0 << 10);
                        return ((prod < 0 ? neg : pos) >> (2 * e)) & 3;
                    }
                    e++;
                }
            return -1;
        }

        // Enters the cell i through its face ef (-1: the face the path entered by, -1 again if there is
        // none): its vertices, relative to that face, and its density.
        __device__ __forceinline__ void tet_enter(const GridView& g, int ef)
        {
            const TetCell& T = g.tcell[i];
            j = ef < 0 ? entering_face(T) : ef;
            bn = T.dens;
            if (j < 0) return;
            int c0, c1, c2;
            clockwise_vertices(j, c0, c1, c2);
            V.load(T.v[j]);
            C0.load(T.v[c0]);
            C1.load(T.v[c1]);
            C2.load(T.v[c2]);
        }

        // One step of the tetra generator: Pluecker exit-face decision with the plane-intersection
        // fallback (TetraMeshSpatialGrid.cpp:719-819); the final segment before the hull is not
        // returned.  Returns as cross() does.  Ends the path where the reference would not terminate:
        // no entering face (all six products zero) or a non-finite position.
        //
        // Bound by the vector memory path: the lanes' cells lie apart, and the eleven loads of a
        // crossing kept the return path busy 92 % of the time.  The vertices therefore stay in
        // registers, ordered as seen from the entering face; the next cell shares three of them, and
        // the record of the face between the two holds the fourth, with all else the crossing needs:
        // four loads of one 64-byte line.  150 000 vertices, 64 instances, 2^20 packets: 79 -> 58 ms.
        static constexpr int kTetReload = -1;  // k where the next cell's vertices do not match
        __device__ __forceinline__ int cross_tetra(const GridView& g, int& m, double& ds, double& n)
        {
            if (j < 0 || !(isfinite(rx) && isfinite(ry) && isfinite(rz)))
            {
                state = kOutside;
                return -1;
            }
            int c0, c1, c2;
            clockwise_vertices(j, c0, c1, c2);
            const double wx = rx - V.x, wy = ry - V.y, wz = rz - V.z;
            const double mx = ky * wz - kz * wy, my = kz * wx - kx * wz, mz = kx * wy - ky * wx;
            const double prod0 = mx * (V.x - C0.x) + my * (V.y - C0.y) + mz * (V.z - C0.z);
            const bool clock0 = prod0 < 0;
            const double qx = clock0 ? C1.x : C2.x, qy = clock0 ? C1.y : C2.y, qz = clock0 ? C1.z : C2.z;
            const double prodi = mx * (V.x - qx) + my * (V.y - qy) + mz * (V.z - qz);
            const bool cclocki = prodi >= 0;
            // dtable {{1,0},{0,2}} indexes the clockwise vertices; which of them lies opposite the exit
            int q = clock0 ? (cclocki ? 2 : 0) : (cclocki ? 0 : 1);
            if (__builtin_expect(prod0 == 0. || prodi == 0., 0))
            {
                q = -1;
                double least = DBL_MAX;
                for (int u = 0; u < 3; ++u)
                {
                    const TetFace& F = g.tface[4 * static_cast<int64_t>(i) + pick3(u == 0, u == 1, c0, c1, c2)];
                    const double ndotk = F.n[0] * kx + F.n[1] * ky + F.n[2] * kz;
                    if (ndotk > 0)
                    {
                        const double d = (F.n[0] * (V.x - rx) + F.n[1] * (V.y - ry) + F.n[2] * (V.z - rz)) / ndotk;
                        if (d < least)
                        {
                            least = d;
                            q = u;
                        }
                    }
                }
                if (q < 0)
                {
                    ask = true;
                    return 0;
                }
            }
            const bool q0 = q == 0, q1 = q == 1;
            const int leaving = pick3(q0, q1, c0, c1, c2);
            TetFaceRec F;
            F.load(g.tface + 4 * static_cast<int64_t>(i) + leaving);
            const double ndotk = F.a.x * kx + F.a.y * ky + F.b.x * kz;
            const double d = (F.a.x * (V.x - rx) + F.a.y * (V.y - ry) + F.b.x * (V.z - rz)) / ndotk;
            if (__builtin_expect(d < g.eps, 0))
            {
                ask = true;
                return 0;
            }
            rx += kx * d;
            ry += ky * d;
            rz += kz * d;
            const int nxt = F.cell();
            if (nxt < 0)
            {
                state = kOutside;
                return -1;
            }
            m = i;
            ds = d;
            n = bn;
            k = 0;
            // the exit face's vertices, then in the next cell's order
            const uint32_t link = F.link();
            const uint32_t p = link >> (4 * j);
            const TetVert X1 = pick_vert(q0, q1, C1, C2, C0), X2 = pick_vert(q0, q1, C2, C0, C1);
            const int p0 = p & 3, p1 = (p >> 2) & 3, p2 = 3 - p0 - p1;
            i = nxt;
            j = (link >> 16) & 3;
            bn = F.d.y;
            if (__builtin_expect((link >> 18) & 1, 0))
            {
                ask = true;
                k = kTetReload;
            }
            const TetVert X0 = V;
            C0 = pick_vert(p0 == 0, p0 == 1, X0, X1, X2);
            C1 = pick_vert(p1 == 0, p1 == 1, X0, X1, X2);
            C2 = pick_vert(p2 == 0, p2 == 1, X0, X1, X2);
            V = TetVert{F.c.x, F.c.y, F.d.x};
            return 1;
        }
    };
}
