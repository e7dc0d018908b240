// Levenberg-Marquardt solve of Deformer::DeformWithRot (deformer.cc:94-171)
// on gfx950: positions and per-vertex angle-axis rotations.
#pragma once

#include "mo_common.h"
#include "mo_lm.h"

namespace mo {

struct RotPairDesc {
  const float* grid;   // N^3 FP32 distance grid of the target
  int N;
  int nv;              // vertices
  int nh;              // half-edges (face edges with distinct endpoints)
  long long vbase;     // offset in the per-vertex arrays
  long long hbase;     // offset in the per-half-edge arrays
  long long lbase;     // offset in the vertex half-edge lists
  float lambda;        // EdgeLossWithRot lambda
};

constexpr int kRotVSlots = 28;   // float4 work slots per vertex
constexpr int kRotHSlots = 7;    // float4 work slots per half-edge

struct RotArrays {
  const float4* x0;    // rest position (normalized frame)
  float4* u;           // displacement from x0 (in/out)
  float4* w;           // angle-axis rotation (in/out)
  const int4* vadj;    // (first list entry, outgoing count, incoming count, 0)
  const int* vlist;    // local half-edge ids: the outgoing ones, then the incoming ones
  const int2* hab;     // local (a, b) of each half-edge, a = F[f][j], b = F[f][j+1]
  float4* vwork;       // kRotVSlots per vertex, slot-major over all vertices
  float4* hwork;       // kRotHSlots per half-edge, slot-major over all half-edges
};

int lm_rot_launch(const RotPairDesc* pairs_dev, int npairs, const RotArrays& arrays, const LMOptionsDev& opt,
                  LMResultDev* results_dev, long long total_vertices, long long total_half_edges, int block_threads,
                  hipStream_t s);

// Multi-workgroup variant (k_lm_rot_team), laid out as lm_team_launch
// (mo_lm.h): wg_dev entries (team, rank, size, -), team t solves problem
// plist[t]; cnt / part / abort_flag as there; coop as for
// lm_rot_chip_launch.
int lm_rot_team_capacity(int block_threads);
int lm_rot_team_launch(const RotPairDesc* pairs_dev, const int* plist, const int4* wg_dev, int nwg,
                       const RotArrays& arrays, const LMOptionsDev& opt, LMResultDev* results_dev,
                       long long total_vertices, long long total_half_edges, int block_threads, int coop,
                       unsigned* cnt, double* part, int* abort_flag, hipStream_t s);

// On-chip solver (k_lm_rot_chip): a problem's vertices are split into chunks
// of at most kRotChip, one workgroup per chunk with one vertex per thread;
// the workgroups of a problem (at most kRotChipTeam) are its team.  A chunk
// reads other chunks' vertices through its halo list.
constexpr int kRotChip = 512;         // largest chunk (two instances: 256 and 512 threads)
constexpr int kRotChipTeam = 64;
constexpr int kRotMaxMult = 63;       // parallel half-edges of one direction merged into one entry

struct RotChunk {
  int pid;             // problem
  int team;            // its slots and, in a launch, its team number
  int rank, size;      // this workgroup in the team
  int lo, own;         // vertices [lo, lo + own) of the problem, own >= 1
  int nhalo, nent;
  long long halo;      // first halo entry
  long long ent;       // first adjacency entry
};

struct RotChipArrays {
  const float4* x0;
  float4* u;                 // out: displacement
  float4* w;                 // in/out: rotation
  const int2* row;           // per vertex: (first entry in its chunk, entries)
  const unsigned* ent;       // record index | out multiplicity << 20 | in multiplicity << 26
  const int* halo;           // vertex (of the problem) behind each halo record
  float4* ev;                // per entry work: rest edge, lambda A^T r, w_i - w_j
  float4* er;
  float4* es;
  unsigned long long* pub;   // per vertex: kRotPubWords published words
};
constexpr int kRotPubWords = 5;

// dynamic LDS of a chunk: records (own and halo), then entries
size_t lm_rot_chip_lds(int threads, int nhalo, int nent);
int lm_rot_chip_capacity(int threads, size_t lds_bytes);   // co-resident workgroups, 0: cannot launch
// slots: kTagSlotWords zeroed 64-bit words per team; coop: 0 when every team
// has one workgroup, else the launch is cooperative, the coop-th such one of
// the call.  Returns kCoopRefused when the runtime refused the grid.
int lm_rot_chip_slot_words();
int lm_rot_chip_launch(const RotPairDesc* pairs_dev, const RotChunk* chunks_dev, int nchunks, const RotChipArrays& a,
                       const LMOptionsDev& opt, LMResultDev* results_dev, int threads, size_t lds_bytes, int coop,
                       unsigned long long* slots, int* abort_flag, hipStream_t s);

}  // namespace mo
