// kernels.hpp -- launchers of the gfx950 kernels (host-callable).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace sgt {

// Scalars the iteration keeps on the device (reductions and Z).
struct DevScalars {
  double minv[4];   // min of the centred Y per dimension
  double maxv[4];   // max of the centred Y per dimension
  double Z;         // normalisation term (sum z_i - N)
  double kl;        // KL divergence (tsneCost)
  double zexact;    // exact-repulsion Z (validation)
  double pad;
  // device clock (wall_clock64) at the starts of an iteration's spread,
  // convolution, gather and update, written by those phases' own kernels, and
  // at the end of the last centring: phases are timed without event packets
  // between the kernels (six timed events cost 19-25 us per iteration)
  unsigned long long stamp[5];
};
enum StampAt { STAMP_S2G = 0, STAMP_CONV = 1, STAMP_G2S = 2, STAMP_UPDATE = 3, STAMP_END = 4 };

// The part of it the host reads every iteration, in pinned memory, written by
// the centring itself: `seq` last, so the host polls one word instead of
// queuing a copy and waiting for an event.
struct HostScalars {
  double minv[4], maxv[4];
  unsigned long long stamp[5];  // iteration start, then the spread's, convolution's, gather's and update's
  unsigned long long seq;
  unsigned long long end;       // end of the centring that was asked for it, once the stream has passed it
};

// Partial-reduction workspace: one slot per block.
struct RedWork {
  double *part;       // [max_blocks * 8]
  int max_blocks;
};

// Grid mapping of one iteration (computed on the host from min/max).
struct GridParams {
  int d;
  int nGrid;        // interpolation intervals + 1 (reference nGridDim)
  int ng;           // grid side = nGrid + 2
  int L;            // FFT length (even 2^a 3^b 5^c >= 2 ng - 1)
  float minv[3];    // min of Y per dimension (grid origin)
  float scale;      // (nGrid - 1) / maxy
  float gmax;       // largest float below nGrid - 1 (clamp)
  float center[3];  // charge shift (bounding-box centre)
  double hgrid;     // grid spacing in embedding units
};

// ---- attractive term (kernels_spmv.hip) ----
int launch_attr_csr_seg(hipStream_t s, int d, int group, int n, const int32_t *rowptr,
                        const int32_t *col, const float *val, const float *Y, float *F);
int launch_attr_csr_seg2(hipStream_t s, int d, int group, int unroll, int n, const int32_t *rowptr,
                         const int32_t *col, const float *val, const float *Y, float *F);
int launch_attr_csr_blk(hipStream_t s, int d, int group, int unroll, int rows_per_block, int n,
                        const int32_t *rowptr, const int32_t *col, const float *val, const float *Y, float *F);
// windowed blocked form: win points of Y around each row range staged in LDS
// chunk-cached blocked form: per row range, nslots chunks of 2^chs points of Y
// staged in LDS (slots[range * nslots + k] = chunk id or -1)
int launch_attr_csr_cc(hipStream_t s, int d, int group, int unroll, int rows_per_block, int chs, int nslots,
                       const int32_t *slots, int n, const int32_t *rowptr, const int32_t *col, const float *val,
                       const float *Y, float *F);
// builds slots: counts is scratch of div_up(n, rows_per_block) * div_up(n, 2^chs) ints
int launch_chunk_cache(hipStream_t s, int n, int rows_per_block, int chs, int nslots, const int32_t *rowptr,
                       const int32_t *col, int32_t *counts, int32_t *slots);
int launch_attr_csr_win(hipStream_t s, int d, int group, int unroll, int rows_per_block, int win, int n,
                        const int32_t *rowptr, const int32_t *col, const float *val, const float *Y, float *F);
// column-localised form: per row block, Y at its distinct columns staged in LDS
int launch_attr_csr_loc(hipStream_t s, int d, int group, int nblk, int cap, const int32_t *brow, const int32_t *bu,
                        const int32_t *ucol, const int32_t *rowptr, const uint16_t *lidx, const float *val,
                        const float *Y, float *F);
int launch_attr_csr_row(hipStream_t s, int d, int n, const int32_t *rowptr, const int32_t *col,
                        const float *val, const float *Y, float *F);
int launch_attr_coo(hipStream_t s, int d, int64_t nnz, const int32_t *row, const int32_t *col,
                    const float *val, const float *Y, float *F);
int launch_attr_ell(hipStream_t s, int d, int n, int width, const int32_t *ecol, const float *eval,
                    const float *Y, float *F);
int launch_kl(hipStream_t s, int d, int n, const int32_t *rowptr, const int32_t *col,
              const float *val, const float *Y, double alpha, const DevScalars *sc, RedWork rw,
              DevScalars *out);

// ---- repulsion (kernels_grid.hip) ----
int launch_fill(hipStream_t s, float *p, int64_t count, float v);
int launch_stream_copy(hipStream_t s, const float4 *in, float4 *out, int64_t count);
// Caller's points (raw [n][d] or [d][n], perm: row -> caller's index, NULL: the
// same) into Y, centred, with min / max into sc and hs; reset: uY = 0, gains = 1.
int launch_set_points(hipStream_t s, int d, int n, const float *raw, int layout, const int32_t *perm, float *Y,
                      int reset, float *uY, float *gains, RedWork rw, DevScalars *sc, HostScalars *hs,
                      unsigned long long seq);
// The reverse for Y or a force, each coordinate times scale (in FP64).
int launch_get_points(hipStream_t s, int d, int n, const float *in, int layout, const int32_t *perm, double scale,
                      float *raw);
// S2G into V [d+1][ng^d] (V is overwritten).  scratch: float workspace for the
// per-block private grids of the LDS path; *needed receives the floats it
// wants (when larger than scratch_floats the global-atomic path runs).
// sc (may be NULL): the phase stamps STAMP_S2G and STAMP_CONV are written to it.
int launch_s2g(hipStream_t s, const GridParams &g, int n, const float *Y, float *V, float *scratch,
               int64_t scratch_floats, int64_t *needed, int mode = 0, DevScalars *stamp = nullptr,
               const int32_t *ord = nullptr);
// Order of the points along the tiles of grid g, for the spread (through ord
// above) and gather of grids no LDS copy holds: key is scratch of n int2, cnt
// of kSpreadBins ints.  Any order gives the same bits; this one gives runs of
// points small windows of the grid.
constexpr int kSpreadBins = 32768;
bool s2g_takes_order(const GridParams &g, int mode);
int launch_spread_order(hipStream_t s, const GridParams &g, int n, const float *Y, int2 *key, int *cnt, int32_t *ord);
int64_t s2g_scratch_need(const GridParams &g, int n, int mode = 0);
// Frep and the partials of Z; *nz receives how many there are:
// launch_update_center adds them up itself, launch_finalize_z puts their sum into sc->Z for others.
int launch_g2s_force(hipStream_t s, const GridParams &g, int n, const float *Y, const float *Phi,
                     float *Frep, int zdirect, RedWork rw, int *nz, DevScalars *stamp = nullptr,
                     const int32_t *ord = nullptr);
int launch_finalize_z(hipStream_t s, int nz, int n, RedWork rw, DevScalars *sc);
int launch_finalize_kl(hipStream_t s, int nblocks, RedWork rw, DevScalars *sc);
// The update of Y from the forces and the nz partials of Z, then the centring
// of the new Y with its min / max into sc and hs (two kernels).  stamp: 1 with the
// phase times, 2 with the iteration's end in hs too.
int launch_update_center(hipStream_t s, int d, int n, float *Y, float *uY, float *gains, const float *Fattr,
                         const float *Frep, float alpha, float momentum, float eta, int nz, RedWork rw,
                         DevScalars *sc, HostScalars *hs, unsigned long long seq, int stamp);
// Device clock now, into sc->stamp[at].
int launch_stamp(hipStream_t s, DevScalars *sc, int at);
int launch_rep_exact(hipStream_t s, int d, int n, const float *Y, float *Frep, RedWork rw,
                     DevScalars *sc);

// ---- FFT convolution (kernels_fft.hip) ----
struct ConvBuffers {
  float2 *W;      // complex work [pairs][...]
  float2 *Kt1;    // (K2, K1) half-spectrum scratch
  float2 *Kt2;
  float2 *Kh;     // (K2^, K1^) half-spectra of the kernels [(L/2+1)^d]
  float2 *tw;     // twiddle tables of every supported length (twiddle_count())
};
int conv_workspace_bytes(int d, int ng, int L, size_t *w_bytes, size_t *k_bytes);
// V [d+1][ng^d] -> Phi [d+1 (+1 with zdirect: K1 * V0 in channel d+1)][ng^d];
// node_major: channels 0-3 of a node as one float4, then channel 4 as a plane
// (what the gather reads; max(4, d + 2) ng^d floats)
int launch_conv(hipStream_t s, const GridParams &g, int zdirect, const float *V, float *Phi,
                const ConvBuffers &b, bool node_major = false);
// twiddle tables of every supported FFT length (twiddle_count() float2)
size_t twiddle_count();
int init_twiddles(hipStream_t s, float2 *tw);
// FFT length of a grid of side ng: smallest even 2^a 3^b 5^c >= 2 ng - 1
int fft_length_for(int ng);

// ---- P construction (kernels_prep.hip) ----
void retain_pool_memory();
// Where the workspaces of the calls below come from: take() gives a block for
// work queued on s from now on, give() takes it back once s has passed the
// work queued so far.  Safe from several threads.
struct ScratchSource {
  virtual int take(hipStream_t s, size_t bytes, void **p) = 0;
  virtual void give(hipStream_t s, void *p) = 0;
  virtual ~ScratchSource() = default;
};
ScratchSource &stream_scratch();  // hipMallocAsync / hipFreeAsync
int launch_knn(hipStream_t s, const float *X, int n, int dim, int k, int32_t *I, double *D, int method,
               int *fallback_rows);
// launch_knn in two halves for callers that must not wait in between:
// knn_begin queues everything up to the certificate and a copy of the count
// of uncertified rows into *count_host (pinned memory for a copy that does
// not block; after a failure knn_release frees what it holds); knn_end, called
// once the stream has passed that copy, queues the exact recomputation of
// those rows and releases the temporaries.
struct KnnPending {
  bool open = false;  // knn_end still has work to queue
  const float *X = nullptr;
  int n = 0, dim = 0, k = 0;
  int32_t *I = nullptr;
  double *D = nullptr;
  int *fb = nullptr;  // device: [0] count, then the rows
  const int *count_host = nullptr;
  ScratchSource *src = nullptr;
  void *ws = nullptr;  // every temporary, one block
};
int knn_begin(hipStream_t s, ScratchSource &src, const float *X, int n, int dim, int k, int32_t *I, double *D,
              int method, int *count_host, KnnPending *kp);
int knn_end(hipStream_t s, KnnPending *kp, int *fallback_rows);
void knn_release(hipStream_t s, KnnPending *kp);  // frees the temporaries without finishing
int launch_perplexity(hipStream_t s, const double *D, int n, int k, double u, float *val,
                      double *beta_out);
int launch_lambda_rescale(hipStream_t s, int n, const int32_t *rowptr, float *val, double lambda,
                          int drop_leaf);
int launch_rowids(hipStream_t s, int n, const int32_t *rowptr, int32_t *row);
int gpu_symmetrize(hipStream_t s, int n, int64_t nnz, const int32_t *rowptr_d,
                   const int32_t *col_d, const float *val_d, int32_t **rowptr_out,
                   int32_t **col_out, float **val_out, int64_t *nnz_out,
                   ScratchSource *out_src = nullptr);
// gpu_symmetrize in two halves (see KnnPending): sym_begin queues the merge of
// P and P^T and a copy of the merged nonzero count into *runs_host; sym_end,
// once the stream has passed that copy, queues the normalisation and the CSR
// build, without waiting for them, into one block of out_src that starts at
// rowptr (nullptr: three hipMalloc'ed arrays).  max_row: the longest row of P when no
// row holds a column twice, else 0 (any P).
struct SymLong {  // its long rows, as the merge lists them
  int *cnt = nullptr;            // [0] rows sorted by a work-group, [1] hubs
  int32_t *mid = nullptr, *hub = nullptr;
  double *part = nullptr;        // of each part of each hub: its sum (after the rows' sums),
  int32_t *end = nullptr;        // and where it ends in the merged row
};
struct SymPending {
  bool open = false;
  int n = 0;
  ScratchSource *src = nullptr;
  void *ws = nullptr;  // the one block the pointers below lie in
  const int32_t *off = nullptr, *rp = nullptr;
  const int32_t *mcol = nullptr;
  const double *mval = nullptr, *total = nullptr;
  SymLong rows;
  const int *runs_host = nullptr;
};
int sym_begin(hipStream_t s, ScratchSource &src, int n, int64_t nnz, const int32_t *rowptr_d, const int32_t *col_d,
              const float *val_d, int max_row, int *runs_host, SymPending *sp);
int sym_end(hipStream_t s, SymPending *sp, int32_t **rowptr_out, int32_t **col_out, float **val_out,
            int64_t *nnz_out, ScratchSource *out_src);
void sym_release(hipStream_t s, SymPending *sp);
int launch_build_ell(hipStream_t s, int n, int width, const int32_t *rowptr, const int32_t *col,
                     const float *val, int32_t *ecol, float *eval, int32_t *tail_cnt);
int launch_build_tail(hipStream_t s, int n, int width, const int32_t *rowptr, const int32_t *col,
                      const float *val, const int32_t *tail_off, int32_t *trow, int32_t *tcol,
                      float *tval);
int device_exclusive_scan(hipStream_t s, const int32_t *in, int32_t *out, int n);
// order[r] = current index of the point placed at r (Morton order of Y over
// the box [lo, lo + extent]^d); inv = order^-1.
int spatial_order(hipStream_t s, int n, int d, int ds, const float *Y, const double *lo, double extent,
                  int32_t *order, int32_t *inv);
int launch_gather_points(hipStream_t s, int n, int ds, const int32_t *order, const float *in, float *out);
int launch_permute_csr(hipStream_t s, int n, int64_t nnz, const int32_t *perm, const int32_t *iperm,
                       const int32_t *rp, const int32_t *col, const float *val, int32_t *rp2,
                       int32_t *col2, float *val2,
                       bool sort_rows = true, bool device_sort = false);

}  // namespace sgt
