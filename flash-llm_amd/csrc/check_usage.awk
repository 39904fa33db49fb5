# Reads the compiler's kernel-resource-usage remarks of one object file and fails (exit 1) when a kernel that the
# launch code's assumptions depend on came out differently:
#   spmm_stream_kernel  every instance must keep two waves per SIMD (the grids are sized for eight waves per CU);
#   spmm_group_kernel   issues its MFMAs as inline assembly on accumulators that must stay where they are: the
#                       build that was verified has 168 VGPRs or fewer and three waves per SIMD (launch bounds);
#                       more registers or a lower occupancy means the compiler started moving accumulators;
#   spmm_wide_kernel    two waves per SIMD, i.e. two workgroups per CU (the choice between it and spmm_group_kernel
#                       counts on them), in 240 VGPRs or fewer (234 in the build that was measured);
#   spmm_quarter_kernel MFMAs as inline assembly on all 256 accumulation registers; few VGPRs (218 in the build that
#                       was measured; 232 with spmm_even_kernel, the same program, at 224) leave no reason to move any;
#   encode_tiles_kernel six waves per SIMD, i.e. six workgroups per CU.
/Function Name:/ { name = $0 }
/ VGPRs: /       { split($0, a, "VGPRs: "); vgprs = a[2] + 0 }
/Occupancy \[waves\/SIMD\]:/ {
    split($0, a, "SIMD]: "); occ = a[2] + 0
    if (name ~ /spmm_stream_kernel/ && occ < 2) { print "spmm_stream_kernel: occupancy " occ " < 2: " name; bad = 1 }
    if (name ~ /spmm_group_kernel/ && (occ < 3 || vgprs > 168)) { print "spmm_group_kernel: " vgprs " VGPRs, occupancy " occ ": " name; bad = 1 }
    if (name ~ /spmm_wide_kernel/ && (occ < 2 || vgprs > 240)) { print "spmm_wide_kernel: " vgprs " VGPRs, occupancy " occ ": " name; bad = 1 }
    if (name ~ /spmm_(quarter|even)_kernel/ && (occ < 1 || vgprs > 232)) { print "spmm_quarter_kernel or spmm_even_kernel: " vgprs " VGPRs, occupancy " occ ": " name; bad = 1 }
    if (name ~ /encode_tiles_kernel/ && occ < 6) { print "encode_tiles_kernel: occupancy " occ " < 6: " name; bad = 1 }
}
END { exit bad }
