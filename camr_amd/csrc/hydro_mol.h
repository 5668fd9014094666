// hydro_mol.h -- the method of lines' hydro source of a whole level.
#pragma once

#include <vector>

#include "canon.h"
#include "hydro_state.h"

namespace camr {

// One box as the kernels see it.
struct MolBox {
    Box bx;
    Canon L;        // layout of q and divu (canon_of(bx))
    double *q;      // compact primitives of grow(bx, 4) (NQC)
    double *divu;   // nodal divergence of bx
    Canon Lu;       // layout of Sborder, dense over grow(bx, 4)
    double *u;      // Sborder (NVAR)
    Arr dsdt;       // dS/dt of bx
    int w, h;       // x-y tile of a block, rim included
    int ntx, nty;   // of them per plane
    int zw, zh;     // x-z tile of a block, rim planes included
    int nzx, ntz;   // of them per row of cells and column
};

// construct_hydro_source of the method of lines (MOL_umeth.cpp:15-142,
// Hydro_umdrv.cpp:57-92) for every box of a level: dS/dt from Sborder,
// written as 0 + the update.  Four launches: primitives, nodal divergence, x
// and y, z with the update.
class MolEngine {
  public:
    MolEngine() = default;
    ~MolEngine();
    MolEngine(const MolEngine &) = delete;
    MolEngine &operator=(const MolEngine &) = delete;
    static bool fits(const Box &bx);
    // ready() afterwards unless memory is short
    int setup(const std::vector<Box> &boxes, const std::vector<Arr> &sb,
              const std::vector<Arr> &dsdt);
    bool ready() const { return tab_ != nullptr; }
    int source(const HydroConst &hc, hipStream_t st, int *status, Prof *prof) const;

  private:
    void release();
    std::vector<MolBox> host_;
    std::vector<int> blk_host_;  // block prefixes: cells, nodes, x-y tiles, x-z tiles
    MolBox *tab_ = nullptr;
    int *blk_ = nullptr;
    double *buf_ = nullptr;
};

} // namespace camr
