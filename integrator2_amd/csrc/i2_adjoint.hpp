// i2_adjoint.hpp -- descriptors of the adjoint kernels (dL/d vertex coordinates).
#pragma once
#include "i2_batch.hpp"

#include <vector>

namespace i2 {

// One mesh as the adjoint kernels see it: the forward pass's outputs they
// need (convergence iteration per ordered task, K per type) and the
// accumulators they write.
struct AdjMesh {
    const i2d::Panel* panels;
    const int64_t* row_start;
    const int64_t* nbr_start;
    const int32_t* nbr;
    const int32_t* lists[2];      // vertex- and edge-sharing (i, j, k), i < j
    const int64_t* off[2];        // where panel i's pairs start in them
    const int64_t* back_start;    // panel j's pairs with earlier panels: 2 k + kind, or -1
    const int64_t* back;
    const int32_t* tri;           // panels' vertices
    const int64_t* inc_start;     // vertices' panels, ascending
    const int32_t* inc;
    int64_t npairs[3];
    const int8_t* conv[3];        // per ordered task, reference task order
    const int* K;                 // refinement iterations per type
    int nT;
    int jtiles;                   // tiles of panels j (disjoint items per block of panels i)
    int niw;                      // wavefronts of 64 panels i
    int jt;                       // panels j per tile
    // Partial cotangents of the panels' vertices, 9 doubles each (vertex a,
    // b, c; x, y, z): ki[tile][i] from the disjoint item (wavefront of i,
    // tile) as the control panel, kj[iw][j] from the wavefront iw of panels
    // i as the influencing panel.  Every slot has one writer.
    double* ki;
    double* kj;
    double* dX;                   // dL/dX, 3 nV (written by the vertex gather)
    double* loss;                 // L (written by the loss gather)
};

// A vertex- or edge-sharing task after its point loop: the cotangents of the
// parameters of its per-point functions and of the panel quantities, for the
// per-task chain to the vertex coordinates (forward-mode dual numbers, one
// coordinate per lane, in a kernel of its own).
struct SingRec {
    int i, j, s1, s2;
    i2d::d3 g[3];       // inner integral: K_j vertices a, b, c
    i2d::d3 cb[5];      // singular context: JB, JC, tau_a, tau_b, tau_c (edge) or JA, tau_a, tau_b, e (vertex)
    double cs;          // 1/|JC - JB| (edge) or 1/sqrt(S_i) (vertex)
    i2d::d3 X[3];       // K_i vertices through the quadrature points
    i2d::q4 F;          // quadrature sum of the regular part
    double fa;          // area of a sub-panel of K_i at the task's level
    i2d::q4 gb;         // the task's (Psi, Theta) cotangent
    double w;           // its weights
    i2d::d3 v;
    double loss;        // the task's term of L
};

// a disjoint item with pairs at reported level >= 2: its pairs are entries base
// to base + n - 1 of the pair list; and such a pair: lane * 32 + bit of its item
// (up to 2,047) and its level
struct DeepItem { int64_t item, base; int n; };
struct DeepPair { int64_t item; int16_t at, level; };
constexpr int N_ADJ_COUNTERS = 5;

struct AdjArgs {
    const AdjMesh* meshes;
    int nmeshes;
    int fixed;
    int last_level;
    int quirk;
    i2d::Rule rule;
    uint64_t seed;
    int64_t disjoint_items;       // items: (mesh, wavefront of 64 panels i, tile of panels j)
    const int64_t* item_base;     // per mesh
    int64_t singular_tasks;       // ordered vertex- and edge-sharing tasks of all meshes
    const int64_t* sing_base;     // [kind * nmeshes + m], kind 0 vertex-, 1 edge-sharing
    unsigned long long* counters; // [0] disjoint item, [1] items with pairs at level >= 2, [2] those pairs, [3] singular tasks at level 2, [4] above
    SingRec* sing_rec;            // per singular task (singular_tasks entries)
    int64_t* sing_deep;           // the singular tasks at level 2 from its start, those above from its end (singular_tasks entries)
    double* sing_dl;              // per singular task: dL/d of its 18 vertex coordinates (I's a, b, c, J's a, b, c)
    double* item_loss;            // per disjoint item: its pairs' terms of L
    double* loss_part;            // per mesh: partial sums of L (k_adj_loss_part)
    uint32_t* deep_mask;          // per disjoint item and lane: bit b set if (i, j0 + b) is at reported level >= 2
                                  // (written for the items in deep_items)
    DeepItem* deep_items;         // the disjoint items that hold such a pair, counters[1] of them
    DeepPair* deep_pairs;         // their pairs, counters[2] of them, as far as deep_cap entries hold an item's
    double* deep_rec;             // per entry: the pair's cotangents
    int64_t deep_cap;
    // the vertex gather: panel sums (9 per panel, mesh m's from pbase[m]),
    // vertices of all meshes (mesh m's from vbase[m])
    double* psum;
    const int64_t* pbase;
    int64_t npanels;
    int64_t nvtx;
    const int64_t* vbase;
};
struct AdjState {
    AdjArgs args{};
    int grid = 0;
    std::vector<int64_t> nV;       // per mesh
    std::vector<int64_t> grad_off; // per mesh: dL/dX (3 nV) then L, in d_grad
    double ms = 0.0;              // device time of the last adjoint run
    int64_t kj_total = 0;         // doubles of K_j slots, all meshes
    DBuf<double> d_grad;          // dL/dX (3 nV) and L
    DBuf<double> d_ki, d_kj;      // partial panel cotangents (all meshes)
    DBuf<double> d_item_loss, d_sing_dl, d_psum, d_loss_part;
    DBuf<int64_t> d_base;         // the base tables of AdjArgs, then the mesh descriptors
    DBuf<uint32_t> d_deep_mask;
    DBuf<DeepItem> d_deep_items;
    DBuf<DeepPair> d_deep_pairs;
    DBuf<double> d_deep_rec;
    DBuf<unsigned long long> d_counters;
    DBuf<SingRec> d_sing_rec;
    DBuf<int64_t> d_sing_deep;
    SideStream* side = nullptr;   // the singular pairs' kernels beside the disjoint pairs' (of the batch or evaluator)
    hipEvent_t e0 = nullptr, e1 = nullptr;
};

void adjoint_release(AdjState*& S);
AdjMesh adjoint_mesh(const i2_mesh* mesh, const int8_t* const conv[3], const int* dK);
int adjoint_setup(AdjState& S, int device, std::vector<AdjMesh> D, const std::vector<const i2_mesh*>& meshes,
                  const i2_integrator* it, uint64_t seed, const int* K = nullptr);
// Enqueues the adjoint kernels (capturable: no host synchronisation, fills by kernels).
int adjoint_launch(AdjState& S, hipStream_t st);
int adjoint_copy_out(const AdjState& S, int mesh, double* loss, double* dLdX);

}  // namespace i2
