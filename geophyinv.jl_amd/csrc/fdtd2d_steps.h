// Several time steps of one 2-D shot per launch (fdtd2d_steps.hip).
#pragma once
#include <memory>

#include "gpi_util.h"

namespace gpi {

// Workgroup tile: rz x wx cells of every array, held for up to `steps` time steps.
struct StepTile {
    int rz, wx, steps;
};

// One workgroup: the cells [z0, z1) x [x0, x1) it updates, and its ranges of the source and
// receiver tables.
struct TileBox {
    int32_t z0, z1, x0, x1, s0, s1, r0, r1;
};

// One source target inside a tile (its halo included): cell = row + rz * column.
struct TileSource {
    int32_t cell;
    int32_t first;       // entries of this cell where this is the first of them, else 0
    int32_t kind;        // 0: both normal stresses (or p), 1: vx, 2: vz
    int32_t target;      // column of the amplitude table
};

// One receiver of a tile: its four taps are cells base, base+1, base+rz, base+rz+1 of an array.
struct TileReceiver {
    int32_t base;
    int32_t array;
    int32_t set;         // index into the record table
    int32_t point;
    float w[4];
};

constexpr int MAX_STEP_REC = 8;
constexpr int MAX_TILE_SOURCES = 256;

struct StepParams2D {
    const float* in[5];      // acoustic p, vx, vz | elastic tauxx, tauzz, tauxz, vx, vz
    float* out[5];
    const float* coef[5];    // at the cells they update: acoustic cx, cz, dtK | elastic cx, cz, dtM, dtlambda, dtavmu
    // CPML memory of the x and z derivatives, velocity update first: elastic dtauxxdx, dtauxzdz, dtauxzdx,
    // dtauzzdz, dvxdx, dvzdz, dvxdz, dvzdx; acoustic dpdx, dpdz, dvxdx, dvzdz
    const float* psi_in[8];
    float* psi_out[8];
    const float* pa[8];      // CPML a, b, kI of each
    const float* pb[8];
    const float* pk[8];
    int ps2[8];              // stride of psi
    int nz, nx, ld, npml;
    uint32_t pml_mask, rigid_mask, free_mask;
    float dxI, dzI, dt;
    int lead;                // halo cells on each side of a tile
    int steps;               // time steps of this launch (lead >= steps * h)
    // arrays that keep every step (their `in` and `out` are slots hstart and hstart + steps): the
    // ring's first slot, else null
    float* hist[5];
    int64_t hslab;
    int hslots, hstart;
    // time reversal (acoustic): before every step p takes stored values on three planes inside
    // the absorbing strips at both ends of each axis (boundary_force!); fx: nt x 6 columns of
    // nz, fz: nt x nx columns of 6, read at fnt - 1 - it; fnp the strips' width per axis (z, x)
    const float* fx;
    const float* fz;
    int64_t fnt;
    int fnp[2];
    int ntile;
    const TileBox* box;
    int64_t it0;
    const TileSource* src;   // sorted by cell within a tile
    const float* amp;        // nt x namp increments of the sources' targets
    int namp;
    const TileReceiver* rec;
    int rnpts[MAX_STEP_REC];
    float* rout[MAX_STEP_REC];
};

// Plan of a shot's launches: tile, coefficients, source and receiver tables, and the second
// state that the launches alternate with.
struct StepPlan {
    int steps = 0;           // most steps of a launch
    int launches = 0;        // kernels per launch of steps: the inner region's tiles and the others
    StepTile tile[2] = {};
    bool inner[2] = {};
    StepParams2D P[2] = {};
    State* st[2] = {};
    std::shared_ptr<State> alt;   // the second of them (its memory in the call's scratch)
    int ders[8] = {};        // derivative fields of psi_in
    int cur = 0;             // state that holds the current wavefield
};

// time steps that one launch takes on this model's grid; 0: such grids are left to the passes
int launch_steps_2d(const Model& m);
// Decides whether the shot (its sources and receivers as planned for the passes) can run
// several steps per launch and prepares it in memory of S; *ok = false leaves it to the passes.
// Without `second` the caller names both states itself.
int plan_steps_2d(gpi_ctx* c, Model& m, Scratch& S, int64_t nt, const Sources& src,
                  const gpi_shot* shot, const std::vector<DevPoints>& rec, StepPlan* plan,
                  bool* ok, bool second = true);
// `steps` <= plan.steps time steps from it0; the arrays of `ring` (if given) take the slots
// after its current one instead of the two states
void run_steps_2d(const Model& m, StepPlan& plan, int64_t it0, int steps, hipStream_t s, Ring* ring = nullptr);

}  // namespace gpi
