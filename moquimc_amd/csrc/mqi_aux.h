// Host-side launchers of the auxiliary kernels (mqi_aux.hip).
#ifndef MQI_AUX_H
#define MQI_AUX_H

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mqi_aux
{
int fill_u64(void* p, unsigned long long v, uint64_t n, hipStream_t s);
// counters of the per-XCD work ranges of a dynamic launch over `total` histories
int queue_init(unsigned long long* q, uint64_t total, hipStream_t s);
int fill_u32(void* p, uint32_t v, uint64_t n, hipStream_t s);
int hu_to_density(const int16_t* hu, float* rho, uint64_t n, float scale, hipStream_t s);
int math_probe(int fn, const double* x, const double* y, double* out, int64_t n, hipStream_t s);
// n_updates FP64 atomic adds to hashed slots of a (n_slots doubles); with
// window > 0 (a power of two below n_slots) the 64 adds of each wave fall in
// one window of that many slots placed at random
int atomic_probe(double* a, uint64_t n_slots, uint64_t n_updates, uint64_t window, hipStream_t s);
int stat_reduce(const double* s1, const double* s2, uint64_t n, double N, float thr, float* d_max, double* d_sum,
                unsigned long long* d_cnt, hipStream_t s);
int scale(double* p, uint64_t n, double w, hipStream_t s);
// dose += w * (stat - snap) outside voxel 0 of each block of nvox
int dose_from_stat(double* dose, const double* stat, const double* snap, uint64_t n, uint64_t nvox, double w,
                   hipStream_t s);
// Dij tables into (voxel; spot, value) lists (mqi_aux.hip): each item's
// maximum and the entries >= rel_thr * max of each of its chunks, then a
// scenario's entries from each chunk's place (start)
int dij_count(const double* vals, const uint64_t* off, uint32_t n_items, uint32_t chunks, double rel_thr,
              double* item_max, uint32_t* counts, hipStream_t s);
int dij_write(const uint32_t* keys, const double* vals, const uint64_t* off, uint32_t item0, uint32_t n_spots,
              uint32_t chunks, const double* item_max, double rel_thr, const uint32_t* start, uint32_t* vox,
              uint64_t* packed, hipStream_t s);
// the tables' entries added to Dose (scenario s at dose + s * stride)
int dose_from_dij(const uint32_t* keys, const double* vals, const uint64_t* off, uint32_t n_items, uint32_t chunks,
                  uint32_t n_spots, uint64_t stride, double* dose, hipStream_t s);
// a CSR's values with their rows: packed[k] = (row, value) of nonzero k
int pack_rows(const int64_t* indptr, const float* val, int64_t n_rows, uint64_t* packed, hipStream_t s);
// stable radix sort of n (key; 64-bit value) pairs by the low `bits` of the
// key; the result is in the tmp arrays if *in_tmp.  With scratch NULL only
// *scratch_bytes is set.
int sort_pairs(uint32_t* keys, uint32_t* keys_tmp, uint64_t* vals, uint64_t* vals_tmp, int64_t n, int bits,
               void* scratch, size_t* scratch_bytes, int* in_tmp, hipStream_t s);
// keys sorted by voxel: the voxels that begin before each tile of MQI_TILE
// keys, and (heads[tiles]) in all
#define MQI_TILE 4096
int tile_heads(const uint32_t* key, int64_t n, uint32_t* heads, hipStream_t s);
// the voxel-major copy of (voxel; spot, value) sorted by voxel, and (spot;
// rank, value) for the sort back; tcol16 or tcol is written
int voxel_rows(const uint32_t* key, const uint64_t* packed, int64_t n, const uint32_t* heads, int32_t* nzvox,
               int64_t* tptr, uint32_t* tptr32, uint32_t* bits, int64_t cols, uint16_t* tcol16, int32_t* tcol,
               float* tval, uint32_t* spot, uint64_t* ranked, hipStream_t s);
int spot_rows(const uint64_t* ranked, const int32_t* nzvox, int64_t n, int32_t* col, int32_t* ccol, float* val,
              hipStream_t s);
// CSR-Adaptive segment sizes (entries of one long-row piece; entries and rows
// of one packed segment)
#define MQI_SEG_LONG 16384
#define MQI_SEG_SHORT 1016
#define MQI_SEG_BUF 1024   // entries of the vectors that cover a packed segment
// entries behind the last one that the products' vectors may cover (zero)
#define MQI_SEG_PAD 4
#define MQI_SEG_ROWS 1024
// rowmap: the element of y each row writes (NULL: row r writes y[r]).  A
// matrix stored without its empty rows (rowmap set) writes y = 0 at the n_y
// elements whose bit in nonempty is clear, from MQI_ZERO_BLOCKS workgroups of
// the same launch (with accumulate it leaves them alone).
// up (device, may be NULL): y = alpha * A x * *up.
#define MQI_ZERO_BLOCKS 1024
int csr_adaptive(const int64_t* indptr, const int32_t* col, const float* val, const float* x, const int64_t* seg_k,
                 const uint32_t* seg_info, int64_t n_seg, const int32_t* split_seg, int64_t n_split, double* part,
                 void* y, int y_is_double, double alpha, const double* up, int accumulate, const int32_t* rowmap,
                 const uint32_t* nonempty, int64_t n_y, hipStream_t s);
// The same over 16-bit columns (D w of a Dij with at most 65536 spots).  From
// MQI_LDS_SEGS segments on its workgroups keep x (n_x entries) in LDS, where
// that leaves room for MQI_LDS_WAVES waves of a CU (24576 entries): 200 spots
// (8.4 M entries) took 43.9 us without and 42.1 with, 150 spots 40.5 without.
#define MQI_LDS 163840   // bytes of LDS of a CU and of a workgroup
#define MQI_CUS 256
#define MQI_LDS_WAVES 8
#define MQI_LDS_SEGS 8192
int csr_adaptive16(const int64_t* indptr, const uint16_t* col, const float* val, const float* x, int64_t n_x,
                   const int64_t* seg_k, const uint32_t* seg_info, int64_t n_seg, const int32_t* split_seg,
                   int64_t n_split, double* part, void* y, int y_is_double, double alpha, int accumulate,
                   const int32_t* rowmap, const uint32_t* nonempty, int64_t n_y, hipStream_t s);
// The quadratic objective of y = alpha * A x on the D w matrices of up to
// MQI_QUAD_MATS scenarios, without y: f[i] = mean over the n_y elements of
// c (y_i - p)^2 (c NULL: 1; f on the device) and, for a single matrix, g =
// 2 / n_y * c (y - p) (float32, when g is set).  terms: n_seg + n_split +
// MQI_QUAD_EMPTY_BLOCKS + MQI_QUAD_SUM_BLOCKS doubles, the terms of the
// segments, of the split rows and (rowmap: the matrix has no empty rows) of
// up to MQI_QUAD_EMPTY_BLOCKS workgroups over the elements whose bit in
// nonempty is clear (y = 0), summed in a fixed order that depends on the
// matrix alone.
#define MQI_QUAD_MATS 16
#define MQI_QUAD_EMPTY_BLOCKS 4096
#define MQI_QUAD_SUM_BLOCKS 256
#define MQI_QUAD_ONE 32768   // terms that one workgroup sums
struct quad_obj {
    const double* p;
    const float*  c;
    float*        g;
    double*       part;   // the segments' terms
    double        two_inv_n;
};
struct quad_mat {
    const int64_t*  indptr;
    const void*     col;
    const float*    val;
    const int64_t*  seg_k;
    const uint32_t* seg_info;
    const int32_t*  split_seg;
    const int32_t*  rowmap;
    const uint32_t* nonempty;
    double *        part, *terms;
    int64_t         n_seg, n_split;
    double          alpha;
    uint32_t        empty;   // workgroups of the elements without a row (set by csr_quadratic)
};
int csr_quadratic(const quad_mat* mats, int n, int cols16, const float* x, int64_t n_x, const double* p,
                  const float* c, float* g, int64_t n_y, double* f, hipStream_t s);
// D^T g over column deltas (mqi_aux.hip): the 16-bit deltas of each row's
// columns (0 at row starts and where a row skips more than 65535 columns,
// those positions listed in gaps), the column before each piece's first
// delta, the pieces restaged lane-major in whole 256-nonzero batches (pb:
// staged starts, n_p + 1 entries) with one byte per delta, deltas of 255
// and more kept in per-piece escape lists (ecount: escapes per piece; ebase:
// their exclusive prefix sums), and the product: one wave per piece into
// part[piece] in the order of the headers, then each row's pieces summed in
// a fixed order.
#define MQI_PIECE 4096          // nonzeros per piece
#define MQI_PIECE_WAVES 8       // waves per workgroup of the product
#define MQI_PIECE_BATCHES 8     // 256-nonzero batches a wave has in flight
int deltas16(const int64_t* indptr, const int32_t* col, int64_t rows, int64_t nnz, uint16_t* dcol,
             unsigned long long* n_gaps, int64_t* gaps, int64_t cap, hipStream_t s);
int piece_base(const int32_t* col, const uint16_t* dcol, const int64_t* pk, int64_t n_p, int32_t* pbase,
               hipStream_t s);
int piece_escapes(const uint16_t* dcol, const int64_t* pk, int64_t n_p, uint32_t* ecount, hipStream_t s);
// esc: the escapes, plus 64 entries of padding the product may read
int stage_pieces(const float* val, const uint16_t* dcol, const int64_t* pk, const int64_t* pb, const uint32_t* ebase,
                 int64_t n_p, float* sval, uint8_t* sd8, uint16_t* esc, hipStream_t s);
// a piece as the product reads it: batches [batch0, batch0 + batches) of
// the staged arrays, the column its first delta adds to, its index, and the
// position of its first escape
struct alignas(16) piece_hdr {
    uint32_t batch0, batches;
    int32_t  base, piece;
    uint32_t esc0, pad[3];
};
int pieces_staged(const float* sval, const uint8_t* sd8, const uint16_t* esc, const float* x, const piece_hdr* hdr,
                  int64_t n_p, const int32_t* row_piece, int64_t rows, double* part, void* y, int y_is_double,
                  double alpha, const double* up, int accumulate, hipStream_t s);
// D^T g on compacted x (float, or double rounded to float): xc = x[nzvox]
int gather_x(const void* x, int x_double, const int32_t* nzvox, int64_t n, float* xc, hipStream_t s);
// grouped scoring: out[s][i] += pair[stride i + s] for s < ns, i < n (stride
// 2 or 4), pair cleared
int pair_fold(double* const* out, int ns, int stride, double* pair, uint64_t n, hipStream_t s);
}   // namespace mqi_aux

#endif
