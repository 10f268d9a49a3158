export TMPDIR=/tmp
timeout -s KILL 60 rocprofv3 --pmc SQ_LDS_BANK_CONFLICT SQ_LDS_IDX_ACTIVE SQ_ACTIVE_INST_VALU SQ_INSTS_VALU SQ_INSTS_LDS SQ_BUSY_CU_CYCLES SQ_WAIT_INST_LDS SQ_VALU_MFMA_BUSY_CYCLES GRBM_GUI_ACTIVE -f csv -d gpurun_out/pmc -o t -- python3 _work/prof.py 1b-select-b16-16k 2 > gpurun_out/pmc.log 2>&1
