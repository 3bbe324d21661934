// Host-side declarations shared by the lcsx translation units (not part of the C ABI).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string>
#include <vector>

namespace lcsx
{

void set_error(const std::string& msg);
#define LCSX_HIP(call)                                                                                     \
    do                                                                                                     \
    {                                                                                                      \
        hipError_t e_ = (call);                                                                            \
        if (e_ != hipSuccess)                                                                              \
        {                                                                                                  \
            ::lcsx::set_error(std::string(#call) + ": " + hipGetErrorString(e_));                         \
            throw ::lcsx::HipFailure();                                                                    \
        }                                                                                                  \
    } while (0)
struct HipFailure
{
};
struct NoDevice
{
};
// A pair or contact list needs more entries than the library's cap (the message says which).
struct CapacityFailure
{
};

template <class T>
struct DBuf
{
    T*     p = nullptr;
    size_t n = 0;
    void   alloc(size_t count)
    {
        free();
        n = count;
        if (count) LCSX_HIP(hipMalloc((void**)&p, count * sizeof(T)));
    }
    void free()
    {
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
    void upload(const T* h, size_t count, hipStream_t s)
    {
        if (count > n) alloc(count);
        if (count) LCSX_HIP(hipMemcpyAsync(p, h, count * sizeof(T), hipMemcpyHostToDevice, s));
    }
    void upload(const std::vector<T>& h, hipStream_t s) { upload(h.data(), h.size(), s); }
    void download(T* h, size_t count, hipStream_t s) const
    {
        if (count) LCSX_HIP(hipMemcpyAsync(h, p, count * sizeof(T), hipMemcpyDeviceToHost, s));
    }
    ~DBuf() { free(); }
    DBuf() = default;
    DBuf(const DBuf&) = delete;
    DBuf& operator=(const DBuf&) = delete;
};

struct NodeBox
{
    float4 lo, hi;  // .w unused
};

// ------------------------------------------------------------------ LBVH
// A forest of independent trees, one per segment (scene of a batch): the leaves of segment g are
// the elements [seg0[g], seg0[g+1]). Leaves are sorted by (segment, Morton key, element), each
// segment's tree is the Karras tree of its own keys, and queries start at their segment's root.
// Node ids: inner nodes [0, ni) with segment g's at [ib_g, ib_g + n_g - 1), then leaves
// [ni, ni + n) in sorted order; with one segment this is the reference's numbering.
struct Lbvh
{
    int               arity = 3;
    uint32_t          n     = 0;  // leaves
    uint32_t          ni    = 0;  // inner nodes: n minus the number of non-empty segments
    const uint32_t*   prims = nullptr;  // device, arity per leaf (not owned)
    uint32_t              nseg = 1;
    std::vector<uint32_t> seg0_h, ib_h, roots_h, cover_h, tab_h;  // per segment (seg0_h: nseg + 1)
    DBuf<uint32_t>    seg_of_leaf, inner_seg, seg_tab, roots, khi[2];
    DBuf<uint32_t>    keys[2], vals[2], hist;
    DBuf<float4>      center;
    DBuf<uint64_t>    morton_sorted;
    DBuf<uint32_t>    parent, object_idx, gbox;
    DBuf<uint2>       children;
    DBuf<NodeBox>     nodes;
    // per inner node: both child boxes with the child codes in the .w lanes (inner child: its
    // node id; leaf child: 0x80000000 | element id), so a traversal step is one 64 B load
    DBuf<float4>      packed;
    DBuf<uint32_t>        scan_tmp;
    // treelet refit: every inner node whose subtree has at most kTreeletLeaves leaves belongs to
    // the treelet of its highest such ancestor; a treelet's inner nodes are a contiguous index
    // range (Karras layout), refit by one workgroup. The inner nodes above the treelets ("top"),
    // sorted by depth, are refit by one workgroup afterwards. tcount: treelets, top nodes.
    DBuf<uint32_t>        tsize, tfirst, tleaf, troots, tcount, top_list, top_depth, top_order, top_level_ptr;
    // per top node (in top_order): its two children's node ids, bit 31 set on a top child, and
    // the top children's indices in top_order (top_idx: node id -> index, top nodes only)
    DBuf<uint4>           top_child;
    DBuf<uint32_t>        top_idx;
    bool                  counted = false;  // ntop and ntreelets were read back (large trees, batches)
    uint32_t              ntop = 0;         // inner nodes above the treelets
    std::vector<uint32_t> top_lvp_h;        // top_level_ptr on the host when ntop > kTopLds
    uint32_t              ntreelets = 0;
    // packed keys: largest element id under each child (false) or largest sorted leaf index
    // (true, for sorted self-queries)
    int                   sorted_keys = 0;
    uint32_t*         sorted_to_orig = nullptr;  // points into vals[?] after construct
    DBuf<uint32_t>    leaf_of;                   // its inverse: the sorted leaf of an element
    // traversal stack entries past a query's LDS part (grown by lbvh_query as needed)
    mutable DBuf<uint32_t> spill;
    // per inner node: the 4-wide record (the slots of both children's packed records; a leaf
    // child is one slot and an empty one), written by the refit (wide_ready)
    DBuf<float4>      packed4;
    bool              wide_ready = false;

    // seg0: nseg + 1 leaf offsets (null: one segment of all leaves)
    void init(int arity_, const uint32_t* device_prims, uint32_t n_leaves, const uint32_t* seg0 = nullptr,
              uint32_t nseg_ = 1);
    // verts_per_seg: vertices of each segment; the global box of segment g covers its first
    // min(n_g, 256 ceil(verts_g / 256)) leaves (lbvh.cpp:958, 968)
    void construct(const float* x, const uint32_t* verts_per_seg, hipStream_t s);
    void finish(hipStream_t s);  // construct, from the sorted leaves on
    // wide: with the 4-wide records
    void refit(const float* x0, const float* x1, const float* pad, hipStream_t s, bool wide = true);
    uint32_t n_inner() const { return ni; }
    uint32_t n_nodes() const { return n + ni; }
};

// Exclusive scan of n counts into out[0..n] (out[n] = total; out may be in), one launch or three.
// tmp holds scan_tmp_words(n) words.
uint32_t scan_tmp_words(uint32_t n);
void     launch_scan_excl_u32(const uint32_t* in, uint32_t* out, uint32_t n, uint32_t* tmp, hipStream_t s);

// Stable LSD radix sort of n entries by the key pair (hi, lo), moving a 32-bit value along: lo, hi
// and val are ping-pong pairs of n-entry buffers, sorted on their low lo_bits / hi_bits bits;
// hist holds sort_hist_words(n) words, tmp scan_tmp_words(sort_hist_words(n)), or those of a larger n
// (neither shrinks as n grows). Returns the index (0 or 1) of the buffers that hold the result.
uint32_t sort_hist_words(uint32_t n);
int      launch_sort_key_pairs(uint32_t* lo[2], uint32_t* hi[2], uint32_t* val[2], uint32_t n, int lo_bits, int hi_bits,
                               uint32_t* hist, uint32_t* tmp, hipStream_t s);

// Query modes for the solver's broad phase.
enum QueryMode
{
    QueryVerts = 0,  // query box per vertex: AABB(x0[i], x1[i]) padded by offset[i] + dhat[i]
    QueryEdges = 1,  // per edge: AABB of both endpoints at x0, x1, padded by offset[e0] + dhat[e0]; keeps e < leaf
    QueryBoxes = 2   // explicit boxes (6 floats each), optional edge filter
};
struct QueryArgs
{
    int             mode;
    uint32_t        n_queries;
    const uint32_t* vert_scene;  // per vertex: segment of the query (null: segment 0)
    const uint8_t*  active;      // per segment: 0 skips its queries (null: all)
    const uint8_t*  row_kind;    // QueryVerts: rows of kind >= 2 (affine-body DOFs) are not points (null: all)
    const float*    x0;
    const float*    x1;
    const uint32_t* edges;
    const float*    offset;
    const float*    dhat;
    const float*    boxes;
    int             edge_filter;
    uint32_t*       pairs;
    uint32_t        capacity;
    uint32_t*       count;
    uint32_t*       overflow;  // set to 1 if a traversal stack overflowed (may be null)
    // QueryEdges on a tree refit with sorted_keys: thread i queries edge order[i] (the sorted
    // leaf order) and keeps the leaves after leaf i; valid when the pair test is symmetric
    // (every vertex has the same offset and the same d_hat)
    int             sorted_self;
    const uint32_t* order;
    // traversal shape (0 .. kQueryVariants - 1; out of range: kQueryDefault): LDS stack entries
    // and per-wavefront pair staging, see kQueryShapes; every shape finds the same pairs
    int             variant = -1;
};
constexpr int kQueryVariants = 10;
constexpr int kQueryDefault  = 7;
constexpr int kQueryElements = 4;  // of vertices and edges against an LBVH, where a shape of boxes only is asked for
void lbvh_query(const Lbvh& t, const QueryArgs& a, hipStream_t s);

// The hierarchy that the solver's broad phases walk in the shapes that share a query among lanes: over
// the elements in a static order that keeps a mesh's neighbours together (Setup::cluster), so its
// topology is made once and only its boxes change. Every scene starts a block of kClusterLeaves positions.
struct ClusterQuery
{
    const uint32_t* order;  // queries (points, or edges), every scene padded with kInvalid to whole wavefronts
    uint32_t        n;      // of them, padding included
    const uint32_t* edges;  // null: points
    const uint32_t* vert_scene;
    const uint8_t*  active;
    const float *   x0, *x1, *offset, *dhat;
    uint32_t*       pairs;
    uint32_t        capacity;
    uint32_t*       count;
};
struct ClusterTree
{
    int              arity  = 3;
    uint32_t         blocks = 0;
    const uint32_t*  prims  = nullptr;  // device, arity per element (not owned)
    DBuf<uint32_t>   elem, scene_block;  // element at a position (kInvalid: none); first block of each scene, and the end
    DBuf<float4>     rec, top;           // records, blocks' boxes
    void init(int arity_, const uint32_t* device_prims, const std::vector<uint32_t>& order,
              const std::vector<uint32_t>& scene_block_, hipStream_t s);
    // leaf_of: the elements' keys (null: their ids)
    void refit(const float* x0, const float* x1, const float* pad, const uint32_t* leaf_of, hipStream_t s);
    void query(const ClusterQuery& a, const uint32_t* leaf_of, hipStream_t s) const;
};
bool query_by_clusters(int variant);  // whether a traversal shape is one of those (Setup::cluster_*_use permitting)

}  // namespace lcsx
