// sphg_kernels.h -- host-side launchers of the kernels in sphg_kernels.hip.
// Each takes the scene table and chunk table of one batch launch; a null
// chunk table is a launch over all chunks of scene 0.
#pragma once

#include "sphg_internal.h"

namespace sphg {

// The two tables (before and after the step's sort) of a lone scene, for the
// kernels that write its stall flag; null pointers: a launch that does not
struct Tables {
    DevScene *a = nullptr, *b = nullptr;
};
// the solvers' loops: DFSPH density and divergence, PCISPH pressure
enum LoopKind { LOOP_DENS, LOOP_DIV, LOOP_PCI };
// A lone scene's sweeps control its loops (`fused`).  Up to kFusedLoopChunks
// chunks each block of a sweep adds up the last one's partials; above that they
// are too many for every block, and launch_loop_end decides after an iteration
// that may be the last (1M particles: 973 -> 960 us a step against finalize
// kernels before the loops and after every iteration).
constexpr int kFusedLoopChunks = 2048;
// Launches of up to so many chunks of 256 particles give a particle 4 lanes
// (figures at the launchers).
constexpr int kQuadChunks = 320;                            // list build
constexpr int kQuadPciChunks = 768, kQuadSideChunks = 208, kQuadPaccChunks = 128;   // PCISPH loop
constexpr int kQuadForcesChunks = 384;                      // forces without cohesion
constexpr int kQuadTensionChunks = 128;                     // WCSPH forces with cohesion
constexpr int kQuadSweepChunks = 384;                       // the DFSPH sweeps, normals, cohesion
// `nchunks` chunks, of kBlock particles, are at most `chunks256` of 256
constexpr bool up_to(int chunks256, int nchunks) { return nchunks * kWaves <= chunks256 * 4; }
// The DFSPH sweeps, normals, cohesion: 4 lanes a particle take a block of 64
// particles ~1/3 of the time, and a sweep lasts as long as the compute units
// (256) with the most blocks.
constexpr bool quad_sweep(int nchunks) {
    const int chunks = (nchunks * kWaves + 3) / 4;   // of 256
    return up_to(kQuadSweepChunks, nchunks) && (chunks * 4 + 255) / 256 <= 3 * ((chunks + 255) / 256);
}

// begin_active: also the start of a WCSPH or PCISPH step, counting the
// scenes whose pressure loop runs in begin_active[0] (null: keys only)
void launch_keys(hipStream_t st, const DevScene* T, const Chunk* C, int nchunks, int* begin_active = nullptr);
// maxChunks: the largest cell-chunk count of one scene; up to
// kScanFusedChunks each final-scan block sums the totals before its chunk
// itself (one launch fewer), above it a per-scene scan of the totals runs; up
// to kScanOneChunks the counts are scanned in one launch.  tables, fused: a
// lone DFSPH scene whose density iterations were launched ahead (k_df_positions)
constexpr int kScanOneChunks = 32;
constexpr int kScanFusedChunks = 1024;
void launch_scan(hipStream_t st, const DevScene* T, const Chunk* CC, int ncellchunks, int nscenes, int maxChunks,
                 Tables tables = Tables{}, int fused = 0);
void launch_scatter(hipStream_t st, const DevScene* T, const Chunk* C, int nchunks);
void launch_rank_reorder(hipStream_t st, const DevScene* T, const Chunk* C, int nchunks);
void launch_bvolume(hipStream_t st, const DevScene* T, int scene, int nb, float* tmp);
void launch_build(hipStream_t st, int method, const DevScene* T, const Chunk* C, int nchunks, int fused = 0);
void launch_normals(hipStream_t st, const DevScene* T, const Chunk* C, int nchunks);
// flags: the non-pressure forces (Flags, adhesion among them) of every scene of
// the launch, or -1 where they differ
void launch_forces(hipStream_t st, int method, int flags, const DevScene* T, const Chunk* C, int nchunks);
void launch_dt(hipStream_t st, const DevScene* T, const Chunk* C, int nchunks);
void launch_df_predict(hipStream_t st, const DevScene* T, const Chunk* C, int nchunks, int fused);
// iter: the number of the loop iteration (mode 1, 2)
void launch_df_vel(hipStream_t st, int mode, const DevScene* T, const Chunk* C, int nchunks, int iter, int fused);
void launch_df_err(hipStream_t st, int mode, const DevScene* T, const Chunk* C, int nchunks, int fused);
// kind: 0 dt, 1 density (before loop), 2 density, 3 divergence (before loop), 4 divergence, 5 PCISPH
void launch_finalize(hipStream_t st, int kind, const DevScene* T, int nscenes, int* active, int nchunks);
// also clears active[0..1] for the divergence solve
void launch_df_positions(hipStream_t st, const DevScene* T, const Chunk* C, int nchunks, int* active, int ahead);
void launch_pci_density(hipStream_t st, const DevScene* T, const Chunk* C, int nchunks, int iter, int fused);
void launch_pci_pacc(hipStream_t st, const DevScene* T, const Chunk* C, int nchunks, int iter, int fused);
void launch_pci_integrate(hipStream_t st, const DevScene* T, const Chunk* C, int nchunks, int ahead);
// loop: LoopKind; end: the end of a step; iter: iterations launched so far; a
// null rec: decides only
void launch_loop_end(hipStream_t st, int loop, int end, const DevScene* T, Tables tables, StepRec* rec, unsigned seq,
                     int iter);
void launch_tell_active(hipStream_t st, const int* active, StepRec* rec, unsigned seq);
void launch_clear_stall(hipStream_t st, Tables tables);
void launch_cube(hipStream_t st, const DevScene* T, const Chunk* C, int n);
void launch_emit(hipStream_t st, DevScene* Tc, DevScene* To, int nscenes, int cells);
// PCISPH boundary method
void launch_pb_bself(hipStream_t st, const DevScene* T, int scene, int nb);
void launch_pb_bdensity(hipStream_t st, int pred, const DevScene* T, int scene, int nb, int iter);
void launch_gather_f3(hipStream_t st, float4* dst, const float* src, const uint32_t* id, int n);
void launch_pb_correct(hipStream_t st, int mode, const DevScene* T, const Chunk* C, int n);
void launch_pb_predcorrect(hipStream_t st, const DevScene* T, const Chunk* C, int n);
void launch_time_advance(hipStream_t st, const DevScene* T, int nscenes);
void launch_clear_overflow(hipStream_t st, const DevScene* T, int nscenes);
void launch_fill_int(hipStream_t st, int* p, int v, long n);
void launch_unsort_f4(hipStream_t st, const float4* src, const uint32_t* id, float* dst, int n, int comps);
void launch_unsort_f1(hipStream_t st, const float* src, const uint32_t* id, float* dst, int n, double offset = 0.0);
void launch_unsort_i1(hipStream_t st, const int* src, const uint32_t* id, int* dst, int n);
void launch_keys3(hipStream_t st, const DevScene* T, int scene, int n, int* dst);
void launch_load_state(hipStream_t st, const DevScene* T, int scene, int n, const float* xyz, const float* vel,
                       const float* k, const float* kv);

}  // namespace sphg
