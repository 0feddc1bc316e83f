/* C ABI of the launch schedule (part of libfasttree_plan.so, host only): vnode lists in, the same
 * computation arranged as block programs for a device out, with the records the kernels start from.
 * The counterpart in the reference is the grid of kernel_bench/fasttree.py:443-479, which leaves
 * order and placement to the hardware's dispatcher.
 */
#ifndef FASTTREE_SCHEDULE_H
#define FASTTREE_SCHEDULE_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef struct ft_schedule ft_schedule;

/* FT_SCHEDULE_ERR_INCOMPLETE: the schedule found does not attend all that the vnodes attend (a fault of
 * the library, never of the arguments). */
enum {
  FT_SCHEDULE_OK = 0, FT_SCHEDULE_ERR_NULL_POINTER = -1, FT_SCHEDULE_ERR_ARGUMENT = -2, FT_SCHEDULE_ERR_MEMORY = -3,
  FT_SCHEDULE_ERR_INCOMPLETE = -4
};

/* The arrays of a schedule, all int32.  The first eight are the lists the decode call takes (the
 * per-request entries end with 32 x -1); then the program table (4 per program), a record of 64 per
 * narrow vnode, 256 per program and 16 per request (layouts: include/fasttree_hip.h; the first two
 * kinds only where kv_entries were given); FT_SCHEDULE_COUNTS: wide vnodes, narrow vnodes, programs,
 * block slots the programs were laid out on, narrow vnodes that belong to programs (none).
 * FT_SCHEDULE_WAVE_RECORDS is filled where the plan is one of whole paths (include/fasttree_hip.h,
 * FT_WHOLE_PATHS), which ft_schedule_tree makes of small trees, else empty. */
enum {
  FT_SCHEDULE_KV_OFFS = 0, FT_SCHEDULE_KV_LENS, FT_SCHEDULE_Q_ENTRIES, FT_SCHEDULE_Q_OFFS, FT_SCHEDULE_Q_LENS,
  FT_SCHEDULE_REQ_ENTRIES, FT_SCHEDULE_REQ_OFFS, FT_SCHEDULE_REQ_LENS, FT_SCHEDULE_PROG_TABLE,
  FT_SCHEDULE_NARROW_TABLE, FT_SCHEDULE_PROG_RECORDS, FT_SCHEDULE_REQ_TABLE, FT_SCHEDULE_COUNTS,
  FT_SCHEDULE_KV_ENTRIES, FT_SCHEDULE_NODE_ASSIGNMENTS, FT_SCHEDULE_WAVE_RECORDS, FT_SCHEDULE_ARRAYS
};

/* Arranges vnode lists.  kv_offs / kv_lens / q_offs / q_lens: one entry per vnode (any order);
 * q_entries: the request of every scratch row; kv_entries: the flat slot list the offsets refer to, or
 * NULL (no records are built then).  group: query heads per KV head.  num_cus: the device's compute
 * units.  *modelled_us: what the model expects of the first-stage launch.
 *
 * Without kv_entries, from head_dim 32 on and beside programs, short vnodes of one run that adjoin may come back as one.  Such
 * lists are for ft_decode_programs / ft_decode_static with the program table and no narrow_table, which contract what rounding the
 * probabilities leaves over; ft_decode serves them too, and rounds slightly more of them than of the lists that went in (against
 * 64 bits 2.895e-4 where 2.890e-4). */
int ft_schedule_create(int64_t num_vnodes, const int32_t* kv_offs, const int32_t* kv_lens, const int32_t* q_offs,
                       const int32_t* q_lens, int64_t num_rows, const int32_t* q_entries, int64_t num_kv_entries,
                       const int32_t* kv_entries, int batch_size, int group, int num_kv_heads, int head_dim, int num_cus,
                       double* modelled_us, ft_schedule** out);

/* The same from a tree instead of vnode lists (arguments as in ft_plan_create, include/fasttree_plan.h;
 * kv_slot_map may be NULL).  Which nodes attend their ancestors' tokens together with their own is
 * decided here, by what each choice makes the device move: a child that stays apart costs one
 * partial result per query head of its requests, written and read back; a child that takes its parent's
 * run along re-reads that run, unless it is the last to leave.  FT_SCHEDULE_KV_ENTRIES holds the flat
 * slot list (it ends with 32 x -1), FT_SCHEDULE_NODE_ASSIGNMENTS the decisions (1: taken along). */
int ft_schedule_tree(int num_nodes, const int32_t* parent, const int32_t* seqlen, const int32_t* num_children,
                     const int64_t* req_offs, const int32_t* req_ids, const int64_t* kv_ptrs, const int32_t* kv_slot_map,
                     int64_t kv_slot_map_len, int batch_size, int group, int num_kv_heads, int head_dim, int num_cus,
                     double* modelled_us, ft_schedule** out);

/* As ft_schedule_tree, with a second decision to weigh (decided: num_nodes entries, 1: taken along, 0 for node 0;
 * the reference planner's, for instance; NULL: none): it is taken where its launch is modelled clearly shorter. */
int ft_schedule_tree_weighed(int num_nodes, const int32_t* parent, const int32_t* seqlen, const int32_t* num_children,
                             const int64_t* req_offs, const int32_t* req_ids, const int64_t* kv_ptrs,
                             const int32_t* kv_slot_map, int64_t kv_slot_map_len, const int32_t* decided, int batch_size,
                             int group, int num_kv_heads, int head_dim, int num_cus, double* modelled_us, ft_schedule** out);

/* As ft_schedule_tree_weighed, for a caller whose room for FT_SCHEDULE_KV_ENTRIES is most_kv_entries entries (-1: any number):
 * no plan of whole paths is made that needs more, as such a plan lists a token once for every leaf below it.  (A plan that
 * lists every token once is made all the same.) */
int ft_schedule_tree_within(int num_nodes, const int32_t* parent, const int32_t* seqlen, const int32_t* num_children,
                            const int64_t* req_offs, const int32_t* req_ids, const int64_t* kv_ptrs,
                            const int32_t* kv_slot_map, int64_t kv_slot_map_len, const int32_t* decided,
                            int64_t most_kv_entries, int batch_size, int group, int num_kv_heads, int head_dim, int num_cus,
                            double* modelled_us, ft_schedule** out);

/* Entries of one array, or -1. */
int64_t ft_schedule_size(const ft_schedule* schedule, int which);

/* All arrays behind one another in dst, each at a multiple of 64 entries: offsets[which] is where
 * array `which` starts.  capacity: entries dst holds (FT_SCHEDULE_ERR_ARGUMENT if too few).  With
 * dst == NULL only the offsets and the entries needed (*total) are written. */
int ft_schedule_pack(const ft_schedule* schedule, int32_t* dst, int64_t capacity, int64_t offsets[FT_SCHEDULE_ARRAYS],
                     int64_t* total);

void ft_schedule_destroy(ft_schedule* schedule);

#ifdef __cplusplus
}
#endif

#endif /* FASTTREE_SCHEDULE_H */
