/* Stands in for the library behind the Python extension: every entry point that the extension calls runs `hook`, as a second
 * thread could while the interpreter's lock is released, and returns its status.  Nothing is launched. */
int (*hook)(void);

#define ENTRY(name) \
    int name(void) { return hook ? hook() : 0; }
ENTRY(mhip_slice_pack)
ENTRY(mhip_slice_unpack)
ENTRY(mhip_slice_pack_many)
ENTRY(mhip_slice_unpack_many)
ENTRY(mhip_buffer_read_into)
ENTRY(mhip_buffer_write_from)
ENTRY(mhip_buffer_transfer_many)
ENTRY(mhip_reduce)
ENTRY(mhip_reduce_scatter)
ENTRY(mhip_stack)
ENTRY(mhip_flat_pack)
ENTRY(mhip_flat_unpack)
ENTRY(mhip_fp8_quantize_bucket)
ENTRY(mhip_fp8_dequant_accumulate_bucket_many)
