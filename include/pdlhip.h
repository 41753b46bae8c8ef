/*
 * pdlhip.h -- C ABI of the MI355X (gfx950) implementation of PDL's
 * broadcast-loop compute path: the PDL::Ops binops, the PDL::Ufunc
 * reductions/scans and PDL::Primitive matmult, driven by a restatement of
 * PDL's broadcast engine, executing as hand-written HIP kernels on ndarray
 * data resident in HBM.
 *
 * Plain C types only (no HIP, torch or Perl types in any signature).  Every
 * pointer named `data` below is a DEVICE pointer obtained from
 * pdlhip_alloc (or any other HBM allocation of the calling process).
 *
 * The entry points replace these reference interfaces (PDL 2.106 sources):
 *   pdlhip_run_<op>      pdl_error pdl_run_<op>(pdl *..., OtherPars)
 *                        generated by lib/PDL/PP.pm:1836-1852, 1998-2014
 *                        (type coercion pdlapi.c:1314-1327, redodims
 *                        pdlapi.c:829-869, output creation
 *                        pdlbroadcast.c:490-523, eager readdata
 *                        pdlapi.c:9-38, 746-827)
 *   pdlhip_readdata      the vtable hook pdl_error (*readdata)(pdl_trans*)
 *                        of lib/PDL/Core/pdl.h.PL:381-403, i.e. the
 *                        PP-generated pdl_<op>_readdata (PP.pm:1922-1927),
 *                        running over a broadcast PDL already planned
 *                        (struct pdl_broadcast, pdlbroadcast.h:18-61)
 *   pdlhip_error         pdl_error (pdl.h.PL:370-379)
 *   pdlhip_pdl           the fields of struct pdl (pdl.h.PL:540-586) a
 *                        readdata reads: datatype, state (PDL_BADVAL,
 *                        PDL_NOMYDIMS), dims, PDL_REPRINCS / PDL_REPROFFS /
 *                        PDL_REPRP of the vaffine view (pdl.h.PL:511-517),
 *                        has_badvalue / badvalue (pdl.h.PL:540-586)
 *   pdlhip_alloc/upload/download
 *                        the data side of pdl_allocdata (pdlapi.c:172-209)
 *                        and the host-sync points of Core.xs
 *                        (get_dataref 1145-1160, upd_data 1163-1184)
 */
#ifndef PDLHIP_H
#define PDLHIP_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define PDLHIP_ABI_VERSION 2

/* Type codes in PDL's promotion order (lib/PDL/Types.pm:27-255).  The device
 * computes in SB..D, and in CF and CD (C99 complex arithmetic) for plus,
 * minus, mult, divide, eq, ne, assgn, conversion, sumover, prodover, cumusumover,
 * cumuprodover and matmult without bad values;
 * LD, CLD and the other complex ops are rejected with an error. */
enum {
  PDLHIP_SB = 0, PDLHIP_B, PDLHIP_S, PDLHIP_US, PDLHIP_L, PDLHIP_UL, PDLHIP_IND,
  PDLHIP_ULL, PDLHIP_LL, PDLHIP_F, PDLHIP_D, PDLHIP_LD, PDLHIP_CF, PDLHIP_CD,
  PDLHIP_CLD, PDLHIP_NTYPES
};

/* pdl state bits (pdl.h.PL:300-330 names) */
#define PDLHIP_NOMYDIMS 0x1 /* null ndarray: the op creates dims, type and data */
#define PDLHIP_BADVAL 0x2   /* the bad-value state flag */
#define PDLHIP_VAFFINE 0x4  /* a virtual-affine view (dims/incs/offs of a slice) */

#define PDLHIP_MAXDIMS 16
#define PDLHIP_MAXBIDS 8 /* broadcast ids per ndarray */

/* pdl_error kinds (pdl.h.PL:370-379) */
enum { PDLHIP_ENONE = 0, PDLHIP_EUSERERROR = 1, PDLHIP_EFATAL = 2 };

typedef struct {
  int32_t error;       /* PDLHIP_ENONE / EUSERERROR / EFATAL */
  const char *message; /* thread-local, valid until the next call on the thread */
} pdlhip_error;

typedef union {
  int8_t A; uint8_t B; int16_t S; uint16_t U; int32_t L; uint32_t K;
  int64_t N; uint64_t P; int64_t Q; float F; double D;
} pdlhip_value;

typedef struct {
  int32_t type; /* type code of value, -1 if none (PDL_Anyval) */
  int32_t pad_;
  pdlhip_value value;
} pdlhip_anyval;

typedef struct {
  int32_t datatype;     /* type code; set by the op for a null (NOMYDIMS) output */
  int32_t state;        /* PDLHIP_* state bits */
  int32_t ndims;
  int32_t has_badvalue; /* per-ndarray bad value in `badvalue` (Bad.pd:165-182) */
  int64_t dims[PDLHIP_MAXDIMS];
  int64_t incs[PDLHIP_MAXDIMS]; /* element strides into `data` (vaffine incs) */
  int64_t offs;                 /* element offset into `data` */
  void *data;                   /* device pointer to the root buffer */
  pdlhip_anyval badvalue;
  /* explicit broadcast ids (pdl->broadcastids, pdl.h.PL:569-570, 579; set by
   * broadcastI, Slices.pd:1819-1898): dims [realdims, broadcastids[0]) are
   * the implicit broadcast dims, [broadcastids[k], broadcastids[k+1]) the
   * dims of explicit id k+1, the last entry is ndims.  nbroadcastids = 0
   * means a plain ndarray (one entry, ndims: pdlapi.c:226-228, 601-602). */
  int32_t nbroadcastids;
  int32_t pad2_;
  int64_t broadcastids[PDLHIP_MAXBIDS];
} pdlhip_pdl;

/* ---- library lifecycle -------------------------------------------------- */
pdlhip_error pdlhip_init(int device);
pdlhip_error pdlhip_shutdown(void);
int pdlhip_abi_version(void);

/* ---- device (HBM) buffers: the data of a pdl --------------------------- */
pdlhip_error pdlhip_alloc(size_t nbytes, void **data);
pdlhip_error pdlhip_free(void *data);
pdlhip_error pdlhip_upload(void *dst_device, const void *src_host, size_t nbytes);
pdlhip_error pdlhip_download(void *dst_host, const void *src_device, size_t nbytes);
pdlhip_error pdlhip_synchronize(void);
/* the hipStream_t every launch of this library is ordered on */
void *pdlhip_stream(void);

/* ---- pdl_run_<op> equivalents ---------------------------------------------
 * Null outputs (state & PDLHIP_NOMYDIMS) are created: dims, datatype and a
 * device buffer from pdlhip_alloc (release with pdlhip_free).  Launches are
 * asynchronous on pdlhip_stream(); errors in planning are returned before any
 * launch.  Ops.pd biops: Pars a(); b(); [o]c(); OtherPars int swap. */
pdlhip_error pdlhip_run_plus(pdlhip_pdl *a, pdlhip_pdl *b, pdlhip_pdl *c, int swap);
pdlhip_error pdlhip_run_mult(pdlhip_pdl *a, pdlhip_pdl *b, pdlhip_pdl *c, int swap);
pdlhip_error pdlhip_run_minus(pdlhip_pdl *a, pdlhip_pdl *b, pdlhip_pdl *c, int swap);
pdlhip_error pdlhip_run_divide(pdlhip_pdl *a, pdlhip_pdl *b, pdlhip_pdl *c, int swap);
pdlhip_error pdlhip_run_gt(pdlhip_pdl *a, pdlhip_pdl *b, pdlhip_pdl *c, int swap);
pdlhip_error pdlhip_run_lt(pdlhip_pdl *a, pdlhip_pdl *b, pdlhip_pdl *c, int swap);
pdlhip_error pdlhip_run_le(pdlhip_pdl *a, pdlhip_pdl *b, pdlhip_pdl *c, int swap);
pdlhip_error pdlhip_run_ge(pdlhip_pdl *a, pdlhip_pdl *b, pdlhip_pdl *c, int swap);
pdlhip_error pdlhip_run_eq(pdlhip_pdl *a, pdlhip_pdl *b, pdlhip_pdl *c, int swap);
pdlhip_error pdlhip_run_ne(pdlhip_pdl *a, pdlhip_pdl *b, pdlhip_pdl *c, int swap);
pdlhip_error pdlhip_run_shiftleft(pdlhip_pdl *a, pdlhip_pdl *b, pdlhip_pdl *c, int swap);
pdlhip_error pdlhip_run_shiftright(pdlhip_pdl *a, pdlhip_pdl *b, pdlhip_pdl *c, int swap);
pdlhip_error pdlhip_run_or2(pdlhip_pdl *a, pdlhip_pdl *b, pdlhip_pdl *c, int swap);
pdlhip_error pdlhip_run_and2(pdlhip_pdl *a, pdlhip_pdl *b, pdlhip_pdl *c, int swap);
pdlhip_error pdlhip_run_xor(pdlhip_pdl *a, pdlhip_pdl *b, pdlhip_pdl *c, int swap);
pdlhip_error pdlhip_run_power(pdlhip_pdl *a, pdlhip_pdl *b, pdlhip_pdl *c, int swap);
pdlhip_error pdlhip_run_atan2(pdlhip_pdl *a, pdlhip_pdl *b, pdlhip_pdl *c, int swap);
pdlhip_error pdlhip_run_modulo(pdlhip_pdl *a, pdlhip_pdl *b, pdlhip_pdl *c, int swap);
pdlhip_error pdlhip_run_spaceship(pdlhip_pdl *a, pdlhip_pdl *b, pdlhip_pdl *c, int swap);
/* Ops.pd:382-397 assgn: a(); [o]b() */
pdlhip_error pdlhip_run_assgn(pdlhip_pdl *a, pdlhip_pdl *b);

/* Ufunc.pd:88-140, 413-613: a(n); [o]b() or b(n) */
pdlhip_error pdlhip_run_sumover(pdlhip_pdl *a, pdlhip_pdl *b);
pdlhip_error pdlhip_run_prodover(pdlhip_pdl *a, pdlhip_pdl *b);
pdlhip_error pdlhip_run_dsumover(pdlhip_pdl *a, pdlhip_pdl *b);
pdlhip_error pdlhip_run_dprodover(pdlhip_pdl *a, pdlhip_pdl *b);
pdlhip_error pdlhip_run_cumusumover(pdlhip_pdl *a, pdlhip_pdl *b);
pdlhip_error pdlhip_run_cumuprodover(pdlhip_pdl *a, pdlhip_pdl *b);
pdlhip_error pdlhip_run_dcumusumover(pdlhip_pdl *a, pdlhip_pdl *b);
pdlhip_error pdlhip_run_dcumuprodover(pdlhip_pdl *a, pdlhip_pdl *b);
pdlhip_error pdlhip_run_average(pdlhip_pdl *a, pdlhip_pdl *b);
pdlhip_error pdlhip_run_daverage(pdlhip_pdl *a, pdlhip_pdl *b);
pdlhip_error pdlhip_run_minimum(pdlhip_pdl *a, pdlhip_pdl *c);
pdlhip_error pdlhip_run_maximum(pdlhip_pdl *a, pdlhip_pdl *c);
pdlhip_error pdlhip_run_minimum_ind(pdlhip_pdl *a, pdlhip_pdl *c);
pdlhip_error pdlhip_run_maximum_ind(pdlhip_pdl *a, pdlhip_pdl *c);
pdlhip_error pdlhip_run_minmaximum(pdlhip_pdl *a, pdlhip_pdl *cmin, pdlhip_pdl *cmax,
                                   pdlhip_pdl *cmin_ind, pdlhip_pdl *cmax_ind);
/* Ufunc.pd:484-540: a(n); indx [o]c(m); OtherPars PDL_Indx m_size => m */
pdlhip_error pdlhip_run_minimum_n_ind(pdlhip_pdl *a, pdlhip_pdl *c, int64_t m_size);
pdlhip_error pdlhip_run_maximum_n_ind(pdlhip_pdl *a, pdlhip_pdl *c, int64_t m_size);

/* Primitive.pd:211-245 matmult: a(t,h); b(w,t); [o]c(w,h) */
pdlhip_error pdlhip_run_matmult(pdlhip_pdl *a, pdlhip_pdl *b, pdlhip_pdl *c);

/* Ops.pd ufuncs, Pars a(); [o]b() (Ops.pd:222-265 `ufunc`): bitnot (~,
 * integer types, :327), sqrt (:328), sin (:329), cos (:330), not (!, :331),
 * exp (:332), log (:333), log10 (:365-381); abs is _rabs (:343-358). */
pdlhip_error pdlhip_run_bitnot(pdlhip_pdl *a, pdlhip_pdl *b);
pdlhip_error pdlhip_run_sqrt(pdlhip_pdl *a, pdlhip_pdl *b);
pdlhip_error pdlhip_run_sin(pdlhip_pdl *a, pdlhip_pdl *b);
pdlhip_error pdlhip_run_cos(pdlhip_pdl *a, pdlhip_pdl *b);
pdlhip_error pdlhip_run_not(pdlhip_pdl *a, pdlhip_pdl *b);
pdlhip_error pdlhip_run_exp(pdlhip_pdl *a, pdlhip_pdl *b);
pdlhip_error pdlhip_run_log(pdlhip_pdl *a, pdlhip_pdl *b);
pdlhip_error pdlhip_run_log10(pdlhip_pdl *a, pdlhip_pdl *b);
pdlhip_error pdlhip_run_abs(pdlhip_pdl *a, pdlhip_pdl *b);

/* Bad.pd elementwise ops.  isbad / isgood: a(); int [o]b() (Bad.pd:343,
 * 387); setbadif: a(); int mask(); [o]b() (:584); setvaltobad: a(); [o]b();
 * OtherPars double value (:639); setnantobad, setinftobad,
 * setnonfinitetobad, setbadtonan: a(); [o]b() (:679, 712, 745, 777);
 * setbadtoval: a(); [o]b(); OtherPars double newval (:808).  The output's
 * bad flag follows the reference ($PDLSTATESETBAD / SETGOOD); setnantobad
 * and its like wait for the stream to learn whether they set any value. */
pdlhip_error pdlhip_run_isbad(pdlhip_pdl *a, pdlhip_pdl *b);
pdlhip_error pdlhip_run_isgood(pdlhip_pdl *a, pdlhip_pdl *b);
pdlhip_error pdlhip_run_setbadif(pdlhip_pdl *a, pdlhip_pdl *mask, pdlhip_pdl *b);
pdlhip_error pdlhip_run_setvaltobad(pdlhip_pdl *a, pdlhip_pdl *b, double value);
pdlhip_error pdlhip_run_setnantobad(pdlhip_pdl *a, pdlhip_pdl *b);
pdlhip_error pdlhip_run_setinftobad(pdlhip_pdl *a, pdlhip_pdl *b);
pdlhip_error pdlhip_run_setnonfinitetobad(pdlhip_pdl *a, pdlhip_pdl *b);
pdlhip_error pdlhip_run_setbadtonan(pdlhip_pdl *a, pdlhip_pdl *b);
pdlhip_error pdlhip_run_setbadtoval(pdlhip_pdl *a, pdlhip_pdl *b, double newval);

/* Slices.pd index / index1d / index2d (Slices.pd:142-220), the non-affine
 * slices whose children flow back into their parent:
 *   pdlhip_run_index     <- pdl_run_index:   a(n); indx ind(); [o] c()
 *   pdlhip_run_index1d   <- pdl_run_index1d: a(n); indx ind(m); [o] c(m)
 *   pdlhip_run_index2d   <- pdl_run_index2d: a(na,nb); indx inda(); indx indb(); [o] c()
 * c = a at the index, broadcast over the other dims.  An index out of range
 * (or bad in bad mode) fails with PDL's message, "Error in index:invalid
 * index %d (valid range 0..%d)" (index1d adds "at pos %d"; index2d names the
 * x- or y-index), for the first such element in PDL's loop order; index1d
 * sets c bad for a bad index instead.
 * pdlhip_writebackdata <- the vtable's writebackdata (pdl.h.PL:381-403),
 * i.e. the op's BackCode: a at the index = c, for a child that was written;
 * pdls in signature order, all existing, a and c of the op's type.  Where
 * indices repeat, the last loop position wins, as in PDL's loop. */
pdlhip_error pdlhip_run_index(pdlhip_pdl *a, pdlhip_pdl *ind, pdlhip_pdl *c);
pdlhip_error pdlhip_run_index1d(pdlhip_pdl *a, pdlhip_pdl *ind, pdlhip_pdl *c);
pdlhip_error pdlhip_run_index2d(pdlhip_pdl *a, pdlhip_pdl *inda, pdlhip_pdl *indb, pdlhip_pdl *c);
pdlhip_error pdlhip_writebackdata(const char *op, pdlhip_pdl **pdls, int npdls);

/* Slices.pd rangeb (Slices.pd:561-1015), the engine of range and indexND:
 *   pdlhip_run_rangeb       <- pdl_run_rangeb(PARENT, CHILD, ind_pdl, size_sv, boundary_sv)
 *   pdlhip_writeback_rangeb <- its writebackdata (the BackCode of EquivCPOffsCode)
 * ind: coordinates along dim 0, broadcast over its other dims (converted to
 * indx); size: nsize values (nsize < 0: undefined, all dims 0 -- single
 * elements); boundary: one letter per dim, the last repeated (f/0 forbid,
 * t/1 truncate, e/2 extend, p/3 periodic, m/4 mirror; "" forbids).  The
 * child (created when null) has the index's broadcast dims, the nonzero
 * sizes, then the parent's dims past the index's length; a truncated or
 * (bad mode) bad element is BAD, else 0.  Errors carry PDL's texts ("Error
 * in rangeb:index out-of-bounds in range (index vector #%ld)" for the
 * first such vector, and MakeComp's size and boundary messages).  A zero
 * extent under extend / periodic / mirror truncates (PDL would divide by
 * zero).  Writeback: where positions meet, the last in PDL's loop wins. */
pdlhip_error pdlhip_run_rangeb(pdlhip_pdl *parent, pdlhip_pdl *ind, const int64_t *size, int64_t nsize,
                               const char *boundary, pdlhip_pdl *child);
pdlhip_error pdlhip_writeback_rangeb(pdlhip_pdl *parent, pdlhip_pdl *ind, const int64_t *size, int64_t nsize,
                                     const char *boundary, pdlhip_pdl *child);

/* No counterpart in the reference: pdlhip_run_<op> for the Ufunc.pd
 * reductions a(n); [o]b() (sumover, prodover, dsumover, dprodover, average,
 * daverage, minimum, maximum, minimum_ind, maximum_ind) for callers that
 * cannot allocate device memory (code under HIP graph capture, tight
 * serving loops).  It allocates nothing: the output must exist and the
 * input and output must already have the types the op computes in (no
 * converted copy), else PDLHIP_EUSERERROR.  Long rows and strided ones keep
 * the partials of their chunks in a 7 MiB array the library reserves on each
 * GPU (any input size fits; a launch that needed more would be refused); the
 * results have the bits of pdlhip_run.  All
 * calls on one GPU share that array: calls that overlap on one GPU (other
 * streams, graphs replayed concurrently) race. */
pdlhip_error pdlhip_run_reduce_noalloc(const char *op, pdlhip_pdl *a, pdlhip_pdl *b);

/* Any of the above by its PDL name (pdls in signature order; otherpars:
 * biops {swap}, *_n_ind {m_size}, setvaltobad / setbadtoval {the double's
 * IEEE bit pattern}, others NULL). */
pdlhip_error pdlhip_run(const char *op, pdlhip_pdl **pdls, int npdls, const int64_t *otherpars);
/* the op's parameter count and how many of them are inputs (the vtable's
 * npdls / nparents), e.g. for a binding that tracks which ndarrays an op
 * writes */
pdlhip_error pdlhip_op_info(const char *op, int *npdls, int *nparents);

/* A list of n independent matmults, item i = matmult(a[i], b[i], c[i]) with
 * the semantics of pdlhip_run_matmult (null c[i] are created).  No
 * reference counterpart: PDL runs such a list as a Perl loop of matmult
 * calls.  mode PDLHIP_LIST_QUEUE: one persistent launch over a device list of
 * (product, tile) items, largest inner dimension first, kernel and tile shape
 * picked per shape class by a timing autotuner and cached (a second launch
 * for products of another layout than most, or of an inner dimension below
 * one 16-byte load); PDLHIP_LIST_EACH:
 * one launch per product (the comparison point).  Items that need a type
 * conversion or bad-value handling run through pdlhip_run_matmult. */
enum { PDLHIP_LIST_QUEUE = 0, PDLHIP_LIST_EACH = 1 };
pdlhip_error pdlhip_run_matmult_list(int n, pdlhip_pdl **a, pdlhip_pdl **b, pdlhip_pdl **c, int mode);

/* A prepared matmult list (no reference counterpart): the entries are
 * planned once as pdlhip_run_matmult_list plans them (outputs created),
 * their items and tile decompositions kept in HBM; each launch then runs
 * the whole list (PDLHIP_LIST_QUEUE: one persistent launch or two,
 * PDLHIP_LIST_EACH: one launch per product) and allocates nothing, so it can
 * be captured in a HIP graph.  Entries with bad values, needing a type
 * conversion or of another type than the first are refused. */
typedef struct pdlhip_mmlist pdlhip_mmlist;
pdlhip_error pdlhip_matmult_list_prepare(int n, pdlhip_pdl **a, pdlhip_pdl **b, pdlhip_pdl **c,
                                         pdlhip_mmlist **handle);
pdlhip_error pdlhip_matmult_list_launch(pdlhip_mmlist *handle, int mode);
pdlhip_error pdlhip_matmult_list_free(pdlhip_mmlist *handle);

/* Ragged lists (no reference counterpart: PDL processes a list of ndarrays
 * of uneven lengths with a Perl loop, one broadcast loop per op per
 * ndarray).  Item i of the list has `ninputs` 1-D ndarrays of one length (or
 * 0-dim scalars, the same slot 0-dim in every item), inputs[i*ninputs + k],
 * at most 6 inputs and 12 nodes.  A prepared list evaluates, per element, a
 * chain of Ops.pd binops held in registers (node n: op applied to operands x,
 * y; an operand k >= 0 is input slot k, k < 0 is the result of node -k-1),
 * each node rounding in the trans type PDL would give it, optionally writes
 * every chain value to values[i] (1-D, the chain's type), then applies
 * `final_op` per item:
 *   sumover, dsumover, average, daverage, minimum, maximum -> outputs[i] 0-dim
 *   cumusumover, cumuprodover (integers, no nodes)          -> outputs[i] 1-D
 *   none (values only)
 * all in a fixed set of launches that allocate nothing, so a run can be
 * captured in a HIP graph.  A null output (PDLHIP_NOMYDIMS) is created with
 * the op's output type; an existing one must have that type and shape.
 * `outputs` may be NULL for "none", `values` is NULL when not wanted.
 * Inputs with the bad-value flag are refused (run those ops per ndarray), as
 * are ndarrays with explicit broadcast ids (here and in pdlhip_chain_prepare
 * and the rangeb entry points). */
typedef struct { int32_t op, x, y; } pdlhip_node;   /* op: PDLHIP_OP_* */
enum {
  PDLHIP_OP_PLUS = 0, PDLHIP_OP_MULT, PDLHIP_OP_MINUS, PDLHIP_OP_DIVIDE, PDLHIP_OP_GT, PDLHIP_OP_LT,
  PDLHIP_OP_LE, PDLHIP_OP_GE, PDLHIP_OP_EQ, PDLHIP_OP_NE, PDLHIP_OP_SHIFTLEFT, PDLHIP_OP_SHIFTRIGHT,
  PDLHIP_OP_OR2, PDLHIP_OP_AND2, PDLHIP_OP_XOR, PDLHIP_OP_POWER, PDLHIP_OP_ATAN2, PDLHIP_OP_MODULO,
  PDLHIP_OP_SPACESHIP
};
typedef struct pdlhip_ragged pdlhip_ragged;
pdlhip_error pdlhip_ragged_prepare(int nitems, int ninputs, pdlhip_pdl **inputs, int nnodes,
                                   const pdlhip_node *nodes, const char *final_op, pdlhip_pdl **outputs,
                                   pdlhip_pdl **values, pdlhip_ragged **handle);
/* The same fused chain over ndarrays that broadcast together (PDL's
 * implicit broadcasting of the chain's binops: dims left-aligned, size-1
 * dims repeat), e.g. c = a*b + a with s = sumover(c) in one pass: `value`
 * receives the chain over all broadcast dims (NULL: not kept), `result` the
 * final op along dim 0 (dims 1.. of the broadcast; scans: all dims).  The
 * handle is run, queried and freed with the pdlhip_ragged_* calls below. */
pdlhip_error pdlhip_chain_prepare(int ninputs, pdlhip_pdl **inputs, int nnodes, const pdlhip_node *nodes,
                                  const char *final_op, pdlhip_pdl *value, pdlhip_pdl *result,
                                  pdlhip_ragged **handle);
pdlhip_error pdlhip_ragged_run(pdlhip_ragged *handle);
/* minimum/maximum: after a run, flags[i] = 1 where item i (a row, for a
 * chain) had no good value (its output holds the bad value and gets PDL's
 * bad-value flag, as Ufunc.pd's minimum sets it); waits for the stream.
 * Other ops: all 0. */
pdlhip_error pdlhip_ragged_badflags(pdlhip_ragged *handle, int32_t *flags);
pdlhip_error pdlhip_ragged_count(pdlhip_ragged *handle, int64_t *nitems);
pdlhip_error pdlhip_ragged_free(pdlhip_ragged *handle);

/* HIP graph capture of work enqueued on pdlhip_stream() (no reference
 * counterpart).  While capturing, device memory comes only from the
 * library's cache (no hipMalloc, no synchronisation): an op whose scratch
 * (float matmult packing, long-row reduction partials, converted copies,
 * created outputs) is not cached fails with PDLHIP_EUSERERROR, so run each
 * op once before capturing it.  Three kinds of op need no earlier run: the
 * partial results of strided reductions, of products cut along t and of long
 * integer scans are allocated (hipMalloc, with the thread's capture mode
 * relaxed) where none are cached; the ops of one graph share them.  Blocks
 * an op releases during the capture stay reserved for the graph until
 * pdlhip_graph_destroy.  Calls that wait
 * for the stream (upload, download, synchronize, ragged bad flags,
 * minimum_n_ind/maximum_n_ind with bad values, list and ragged prepare) are
 * refused during a capture.  The handle from pdlhip_graph_end is the
 * library's own (not a hipGraphExec_t). */
pdlhip_error pdlhip_graph_begin(void);
pdlhip_error pdlhip_graph_end(void **graph);
pdlhip_error pdlhip_graph_launch(void *graph);
pdlhip_error pdlhip_graph_destroy(void *graph);

/* How float and double matmult compute (no reference counterpart: the
 * reference has a single scalar loop, Primitive.pd:211-245):
 *   SPLIT16   default; double: FP64 MFMA from 8 per side; float: by its
 *             sizes alone, either FP32 MFMA with sums in parts of a few k
 *             (from 8 per side), or an FP16 hi/lo split, 3 MFMA products,
 *             FP32 accumulate (products with 33..64 per side; and single
 *             ones with sides from 64 and 32 k up, where that is estimated
 *             to be faster, from about 7e9 operations, or beyond 3e10);
 *             sides below 8 as FP32
 *   FP32      plain SIMT kernel with fused multiply-add (float and double)
 *   PDLORDER  SIMT, multiply then add in ascending t: bit-identical to the
 *             reference's loop
 *   FP8       opt-in e4m3 MFMA with per-row/column scales (float) */
enum { PDLHIP_MM_SPLIT16 = 0, PDLHIP_MM_FP32 = 1, PDLHIP_MM_PDLORDER = 2, PDLHIP_MM_FP8 = 3 };
pdlhip_error pdlhip_set_matmult_precision(int mode);
int pdlhip_get_matmult_precision(void);

/* ---- readdata-level entry (a PDL vtable's readdata hook) ------------------
 * PDL has already coerced types, planned the broadcast (initbroadcaststruct)
 * and created outputs; this runs the op over that plan in one launch.  The
 * struct holds the pdl_broadcast fields a PP readdata reads
 * (pdlbroadcast.h:18-61; incs[d*npdls + p] as PDL_BRC_INC) and the core
 * ind_sizes / inc_sizes of the trans (pdl.h.PL:471-503).  A CPU pthread
 * split in PDL's plan is ignored: the whole broadcast is one launch. */
typedef struct {
  int32_t npdls;
  int32_t ndims;
  int64_t dims[PDLHIP_MAXDIMS + 2];
  int64_t incs[(PDLHIP_MAXDIMS + 2) * 6];
  int64_t offs[6];
  int64_t ind_sizes[4];
  int64_t inc_sizes[6 * 2]; /* inc_sizes[p*2 + j]: pdl p, core dim j */
} pdlhip_broadcast;

pdlhip_error pdlhip_readdata(const char *op, int datatype, int bvalflag,
                             const pdlhip_broadcast *brc, pdlhip_pdl **pdls,
                             const int64_t *otherpars);

/* Autotuner (no reference counterpart; PDL picks its CPU split with a
 * static rule, pdlbroadcast.c:95-159).  Kernel variants (list tiles, float
 * GEMM block shapes) are timed once per shape class and kept in
 * $PDLHIP_TUNE_FILE (default
 * ~/.cache/pdlhip/tune-<arch>.txt); PDLHIP_TUNE=0 keeps the default rules.
 * The block shapes of a product all give the same bits; the kernels of a list
 * differ within the bounds of its precision mode.
 * The counts of choices this process measured and reused from the file. */
pdlhip_error pdlhip_tune_stats(int64_t *measured, int64_t *reused);

/* Dry run (no reference counterpart): plan, type-coerce and create output
 * dims/types exactly as the run_<op> calls do, but allocate and launch
 * nothing (data stays NULL).  Needs no device; for host-side tests of the
 * planner. */
pdlhip_error pdlhip_set_plan_only(int enable);

/* ---- measurement ------------------------------------------------------------ */
/* Elapsed milliseconds between two points recorded on pdlhip_stream(). */
pdlhip_error pdlhip_timer_start(void);
pdlhip_error pdlhip_timer_stop(float *ms);
/* Events on pdlhip_stream() for timing single ops inside a longer timed
 * region without synchronising in between. */
pdlhip_error pdlhip_event_create(void **ev);
pdlhip_error pdlhip_event_record(void *ev);
pdlhip_error pdlhip_event_elapsed(void *ev_start, void *ev_end, float *ms);
pdlhip_error pdlhip_event_destroy(void *ev);
/* ---- PDL's random numbers ----------------------------------------------
 * One xoshiro256+ stream seeded as pdl_srand seeds it
 * (Primitive-xoshiro256plus.c:28-43, 111-138), the stream PDL draws with
 * autopthread off (with pthreads PDL gives each thread its own state).  Each
 * element of the existing output, in PDL order (dim 0 fastest, through its
 * dims/incs/offs), takes the next draw pdl_drand = (x >> 11) * 2^-53, and the
 * stream moves on by the element count, across calls as PDL's does.
 *   pdlhip_srandom   <- pdl_run_srandom (Primitive.pd:2113-2140)
 *   pdlhip_run_random  <- pdl_run_random (Primitive.pd:2142-2179): the draw,
 *                         converted to a's type
 *   pdlhip_run_randsym <- pdl_run_randsym (Primitive.pd:2181-2219): the same
 *                         draw; PDL redraws an exact 0.0 (probability 2^-53),
 *                         the device fails the call with PDLHIP_EFATAL instead
 *   pdlhip_grandom   <- PDL::grandom (Primitive.pd:2256-2261) =
 *                       ndtri(randsym(a)) in a's type, float or double only;
 *                       ndtri is PDL::Math's Cephes routine (Math.pd:346-356)
 * Before any srandom the stream is seeded from the clock (PDL_MAYBE_SRAND,
 * Primitive.pd:2095-2097).  These calls read the stream state on the host
 * and fail with PDLHIP_EUSERERROR during a graph capture.
 * pdlhip_rand_state returns the state (4 words) the next draw starts from;
 * pdlhip_rand_skip moves the stream on by n draws, as n elements of random
 * would (no reference counterpart: PDL can only draw them). */
pdlhip_error pdlhip_srandom(uint64_t seed);
pdlhip_error pdlhip_run_random(pdlhip_pdl *a);
pdlhip_error pdlhip_run_randsym(pdlhip_pdl *a);
pdlhip_error pdlhip_grandom(pdlhip_pdl *a);
pdlhip_error pdlhip_rand_state(uint64_t state[4]);
pdlhip_error pdlhip_rand_skip(uint64_t n);

/* Counter-based uniform[lo,hi) fill on the device (splitmix64 of seed+index),
 * for synthetic inputs at sizes a host-side generator cannot supply fast. */
pdlhip_error pdlhip_fill_uniform(pdlhip_pdl *p, uint64_t seed, double lo, double hi);
pdlhip_error pdlhip_fill_normal(pdlhip_pdl *p, uint64_t seed, double mean, double sd);

#ifdef __cplusplus
}
#endif
#endif /* PDLHIP_H */
